// Streaming prefill attention for gfx950: head sizes 64, 128 and 256, no explicit mask, K / V readable in whole
// blocks of 32 keys (dense, or paged with a block size that is a multiple of 32).  The matrix pipe bounds it at 128 and 256:
// 16 / 32 v_mfma_f32_32x32x16_bf16 per block of 32 keys and wavefront, with the vector work of the softmax
// between them.  At 64, where there are 8, that vector work does (busy 58 % of the time, the matrix pipe 39 %, either 78 %).
//
// The work split: four wavefronts of 32 query rows share K / V in LDS, four consecutive (row block, head) pairs of a KV head
// (row_blocks in prefill_common.h); where a group's workgroups run say workgroup_place and spreads_groups.  Five heads per KV head, 40 / 8 of 128: 6 x 32
// rows behind 7232 tokens 140 -> 60 us, 2 x 1152 tokens 50 -> 43, 1 x 256 behind 1216 26.9 -> 26.6 (28.9 with a KV head's workgroups on one XCD).  The whole life of a workgroup behind its address set-up is one block of
// assembly, written by gen_prefill_stream.py, which documents the schedule and the state on entry.
// Against the compiler-scheduled loop of prefill.hip on the same shapes (a whole pass): window of 1024
// keys, 2 x 4096 tokens, 32 / 8 heads 160 -> 137 us; 4 x 2048 tokens, 16 / 16 heads 118 -> 98 us and 16 / 8
// heads 99 -> 83 us; 2 x 2048 tokens, 40 / 8 heads 126 -> 103 us; 2 x 512-token chunks behind 4096 tokens,
// 16 / 16 heads 103 -> 81 us.  Head size 64: 6 x 1280 tokens of 64 / 8 heads 150 -> 116 us, 6 x 2048 in a window of 512
// 184 -> 137, 4 x 1216 behind 2240 of 8 / 8 80 -> 65, a prompt of 32 5.8 -> 4.4; 256, 16 / 8 heads: 2 x 2656 in a window of 1024
// 188 -> 131, 4 x 1216 behind 2240 343 -> 259, a prompt of 32 12.2 -> 7.6.
//
// A launch of few row blocks over many keys (the chunk of one request far into its sequence: 128
// workgroups for 512 rows of 32 / 8 heads, on 256 CUs that hold two each) is split over the keys:
// several workgroups per row block, each with a share of the 32-key blocks, hand float accumulators
// to prefill_merge_kernel.  512 rows behind 8192 tokens: blocks of 64 139 -> 80 us for the pass, blocks of 32
// 231 -> 81 us (unsplit on the plain loop before); 256 rows of 16 / 16 heads behind 8192 228 -> 67 us.  Blocks
// of 32 alone, where nothing is split: 4 x 512 rows behind 4096 tokens 180 -> 144 us.
#include "prefill_stream_kernel.h"

namespace ttpa {

// The line lies where the loop's unit does: whole blocks of 32 keys that lie in one piece.  A dense K / V that ends inside a block, smaller cache blocks,
// windows over a paged cache and explicit masks are the plain loop's.  Wherever both run, this one is
// faster (above) or equal, but for launches at head size 64 that are split and in which half of the wavefronts or more have no rows (one or two
// (row block, head) pairs in a group): over few keys, while the groups are few, the other loop's parts start and end sooner, and with one pair
// two workgroups of a CU, which wait for memory together, hold longer tiles there.  us per pass, this loop / the other: 8 / 8 heads, 1 x 32 rows behind
// 256 tokens 11.4 / 11.0, 1 x 64 behind 512 12.5 / 12.2, 4 x 32 behind 1024 13.0 / 12.5, 6 x 64 behind 512 14.1 / 13.6, 16 / 8, 4 x 32 behind 512 13.3 / 12.9;
// two on a CU: 5 x 32 behind 8192 26.2 / 24.5, 12 x 32 behind 4096 28.2 / 26.8.  Beyond: not split, 1 x 32 behind 64 7.7 / 9.2, 5 x 64 behind 256 10.7 / 12.5;
// more keys, 1 x 32 behind 2048 13.0 / 13.4, 4 x 64 behind 8192 26.1 / 28.6; more groups, 8 x 64 behind 512 14.3 / 14.6; more pairs, 1 x 96 behind 256 11.8 / 13.1.
// (And the block of assembly steps from row to row of the queries and of the output by an unsigned 32-bit number of bytes: rows in descending order or
// further apart are the plain loop's, which has 64 bits for them.)
bool stream_serves(const PrefillArgs &a, int head_size) {
  if (!a.stream || a.mask != nullptr) return false;
  for (const int64_t rows : {a.q_ts, a.out_ts})
    if (rows < 0 || rows >= (int64_t)1 << 31) return false;
  if (!a.pt) return a.skv % kBlockKeys == 0;
  if (a.bs % kBlockKeys != 0 || a.window != 0) return false;
  if (head_size != 64 || a.sq > 2 * kRowsPerWave) return true;
  const int heads = head_group_size(a, head_size), pairs = (a.sq + kRowsPerWave - 1) / kRowsPerWave * heads;
  const bool few_keys = a.keys_bound < 1536 && (int64_t)a.batch * (a.hq / heads) <= 48;
  if (pairs > 2 || !(few_keys || pairs == 1)) return true;
  const Cut c = cut(a, heads, stream_split(head_size));
  return c.parts == 1 || !(few_keys || (c.part >= kSharedPartBlocks && c.workgroups > a.cus));
}

int64_t stream_part_bytes(const PrefillArgs &a, int head_size) {
  return a.pt && stream_serves(a, head_size) ? part_bytes(a, head_group_size(a, head_size), stream_split(head_size), head_size) : 0;
}

// Whether a block-float-8 pass reads bfloat16 copies, written by a launch in front of it, or expands blocks on their way into
// LDS (mode 4).  A block that one workgroup reads is expanded no more often in mode 4, and the copies are a trip through memory:
// they pay where they are few, where they let the keys be split, and where several workgroups read a block of many: two if the keys
// are 512, three if mode 4 is not split itself, four if it is.  us per pass, copies / mode 4: 16/16 heads, 1 x 128 rows behind 128 tokens
// 17.2 / 18.0, 16/8 16.3 / 17.6, 5 x 64 of 16/8 17.8 / 16.7; 40/8 heads (five readers), 5 x 64 behind 128 20.6 / 17.6, 256 24.9 / 22.3, 576 31.1 / 34.4,
// 1024 37.9 / 50.7; 8 x 128 behind 256 34.4 / 32.5, 576 42.3 / 47.3; two row blocks, 8 x 128 of 16/8 behind 128 22.7 / 21.3, 8 x 256 of 16/16
// behind 512 47.8 / 49.1; where mode 4 is split, 24/8 heads, 4 x 64 behind 576 30.2 / 27.8, 40/8, 5 x 64 behind 1984 56.6 / 62.9.
// Not where mode 4 is split and a block is read by at most two workgroups (row blocks times head groups of a KV head):
// 1 x 32 rows behind 512 tokens, 64 / 8 heads 23.1 / 18.8; 4 x 32 rows of 32 / 8 behind 1024 32.1 / 25.3, 4096 49.3 / 38.7; 8 x 128 of 16 / 16 behind
// 4096 167 / 75.6; two row blocks: 4 x 64 of 32 / 8 behind 512 29.5 / 24.9, 8 x 256 of 16 / 16 behind 4096 195 / 128.  Four workgroups: 2 x 64 of
// 64 / 8 behind 4096 49.5 / 55.6; three: 2 x 96 of 32 / 8 46.7 / 50.0.
// At head size 64 mode 4 costs less per block and the copies as much: from eight workgroups per head group on, where the launch has 64.  8 / 8 heads,
// 1 x 1024 rows behind 512 tokens 22.1 / 24.7, 4 x 1024 35.1 / 49.2; 64 / 8, 1 x 256 behind 2048 35.1 / 41.0, 8 x 448 behind 64 42.6 / 63.6; 8 / 2, 5 x 256
// behind 512 21.7 / 21.9, 4 x 256 behind 64 13.9 / 16.1, 192 15.6 / 17.7, 768 21.4 / 21.5, 8192 43.2 / 51.9, but behind 320 and 512 19.1 / 18.8 and 20.4 / 19.9 (16 / 8
// 1 x 512, with as many workgroups and blocks read as often, 19.5 / 20.1 there: no line in these numbers parts the two); below either line: 8 / 8,
// 4 x 256 behind 512 21.8 / 20.7, 8192 56.6 / 50.4; 64 / 8, 8 x 128 behind 512 31.3 / 29.5; 8 / 2, 1 x 512 behind 512 18.8 / 17.6, 1 x 256 behind 8192 30.3 / 28.3.
// (Launches below the line that are large and not split would gain: 8 / 8, 8 x 448 behind 512 28.2 / 33.5, 2048 54.4 / 56.4.)
bool stream_expands(const PrefillArgs &a, int head_size, int64_t room) {
  if (!stream_serves(a, head_size) || head_size == 256) return false;
  if (head_size == 64) {
    const int heads = head_group_size(a, head_size), per_group = ((a.sq + kRowsPerWave - 1) / kRowsPerWave * heads + 3) / 4;
    if (per_group < 8 || (int64_t)a.batch * (a.hq / heads) * per_group < 64) return false;
    // a caller's scratch may hold mode 4's parts, but not the copies and the parts behind them: unsplit copies are the slower form (4 x 256 rows of 8 / 2 behind
    // 8700 tokens, the operator with that scratch, 123 us, mode 4 split 55)
    const int64_t parts = plain_part_bytes(a, head_size, true);
    return parts == 0 || parts > room || expand_bytes(a.batch, a.w, a.hkv, a.bs, head_size) + stream_part_bytes(a, head_size) <= room;
  }
  const int hpw = heads_per_workgroup(a), rows = kRowsPerWave * 4 / hpw;
  const int64_t row_blocks = (a.sq + rows - 1) / rows, readers = row_blocks * (a.hq / hpw / a.hkv);
  const int64_t parts = plain_part_bytes(a, head_size, true);
  const bool splits = parts > 0 && parts <= room;
  // (a table has room for more keys than the chunk's: 8192 rows of it)
  const bool few = a.batch * a.keys_bound * a.hkv <= (a.keys_known ? 5120 : 8192);
  const bool pays = (row_blocks > 1 && (readers > 2 || a.keys_bound >= 512)) || few || part_bytes(a, head_group_size(a, head_size), stream_split(head_size), head_size) > 0 || (readers > (splits ? 3 : 2) && a.keys_bound >= 512);
  return pays && !(splits && readers <= 2);
}

int launch_stream_wide(const PrefillArgs &a, hipStream_t st) { return launch_form<128, kDenseWide>(a, st); }

int launch_stream(const PrefillArgs &a, int head_size, hipStream_t st) {
  switch (head_size) {
    case 64: return launch_stream_d64(a, st);
    case 128: return launch_stream_d<128>(a, st);
    default: return launch_stream_d256(a, st);
  }
}

}  // namespace ttpa
