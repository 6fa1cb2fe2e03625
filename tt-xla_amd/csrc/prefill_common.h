// What the two prefill kernels (prefill.hip: the compiler-scheduled loop; prefill_stream.hip: the
// hand-scheduled one) share: the arguments, the LDS swizzle of a K / V tile and the cache fill that
// rides along with a dense launch.
#pragma once

#include "common.h"

#include <algorithm>

namespace ttpa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));

constexpr int kKeysPerTile = 64;
constexpr int kRowsPerWave = 32;

// x / d for 0 <= x < 2^31 without a division, which is a chain of about 30 vector instructions also where all operands are scalar, and without
// a branch: magic = floor(2^32 / d) (one less for d = 1) gives the quotient or one less.  The set-up of a workgroup has eight of them, two behind
// each other in front of its first request (a chunk of 32 rows behind 256 tokens, 8 / 8 heads of 64: 11.8 -> 11.2 us a pass).
struct Divisor {
  int d;
  uint32_t magic;
};
inline Divisor divisor(int d) { return {d, d > 1 ? (uint32_t)((1ull << 32) / (uint32_t)d) : ~0u}; }
__host__ __device__ __forceinline__ int quotient(const Divisor &v, int x) {
  const uint32_t q = (uint32_t)(((uint64_t)(uint32_t)x * v.magic) >> 32);
  return (int)(q + ((uint32_t)x - q * (uint32_t)v.d >= (uint32_t)v.d ? 1u : 0u));
}

struct PrefillArgs {
  uint16_t *out;
  int64_t out_bs, out_hs, out_ts;
  const uint16_t *q;
  int64_t q_bs, q_hs, q_ts;
  const uint16_t *k, *v;
  int64_t kv_bs, kv_hs, kv_ts;  // dense form
  const int32_t *pt;            // paged form when non-null
  int64_t pt_rs;
  const int32_t *chunk_start;
  const uint16_t *mask;
  int64_t mask_bs, mask_rs;
  int batch, hq, hkv, sq, skv, bs, w, nb, causal;
  uint32_t bs_magic;  // floor(2^32 / bs) + 1: key / bs = mulhi(key, bs_magic) while key * bs < 2^32 (bs >= 2)
  // Dense form with a cache fill in the same launch (fill_kc != null): k / v are also written
  // to the paged caches through fill_pt, by workgroups n_attn ... of the grid.  bs / nb /
  // bs_magic describe the caches; table row of batch entry i = fill_bidx[i] (or i == 0).
  uint16_t *fill_kc, *fill_vc;
  const int32_t *fill_pt;
  int64_t fill_pt_rs;
  const void *fill_bidx;
  int fill_bidx_i64, fill_rows;
  // Grid layout with a fill: fill_groups super-groups of (8 * attn_per_fill attention
  // workgroups, then 8 fill workgroups), then the remaining attention workgroups.  Groups of 8
  // keep an attention workgroup's index congruent to its hardware index modulo 8 (its XCD).
  int fill_groups, attn_per_fill, n_fill;
  int window;  // > 0 (causal only): row i attends keys offset + i - window < j <= offset + i
  float scale_log2e;
  int kv_bfp8;  // paged form: the caches are block-float-8 (mode 4, or expanded into `expand` first)
  void *expand; // scratch for bfloat16 copies of the block-float-8 blocks of this pass, or null
  int spread;   // workgroup_place: every head group over all XCDs
  // The streaming kernel: workgroups per (batch entry, head group), each taking one or several row blocks
  int spg;
  Divisor by_spg, by_groups, by_group_heads;  // spg, head groups of a batch entry, query heads of a KV head
  // The place of a workgroup (workgroup_place): head groups (batch entries times the groups of one), of which whole rounds of eight
  // are dealt to one XCD each and the rest over all of them, group by group if `spread`; query heads of a group
  int full_rounds, rest, head_group;
  Divisor by_rest, by_head_group;
  int spg_even; // > 0: when the row blocks weigh about the same, only this many of them work (equal shares)
  // ... with keys of 128 + 64 features: the second part of q and k, and V's own strides
  const uint16_t *q2, *k2;
  int64_t q2_bs, q2_hs, q2_ts, k2_bs, k2_hs, k2_ts, v_bs, v_hs, v_ts;
  // ... and, paged, several workgroups per row block, each with a part of the keys (scratch from the caller or null)
  float *part_acc;
  int64_t part_bytes;
  int parts, parts_one;  // shares of the keys at most; with one workgroup per CU
  Divisor by_parts, by_parts_one;
  int split_from;        // launches whose last row block has fewer 32-key blocks are not split
  int part_min;          // 32-key blocks of a part at least
  // The host's alone: what the launch is laid out for (set_parts)
  int64_t keys_bound;    // keys of the last row at most, as far as the host knows
  int keys_known;        // ... from the caller, and not from the page table's room
  int cus;               // CUs of the device: asked for once per pass, whose rules need it several times
  int stream;            // 0: the plain loop whatever the shape (TTPA_PREFILL_STREAM=0)
};

// key / block_size without a division instruction sequence (about 30 instructions each, and the
// paged tile loads need several per tile).
__device__ __forceinline__ int div_block(const PrefillArgs &a, int key) {
  return a.bs == 1 ? key : (int)__umulhi((uint32_t)key, a.bs_magic);
}

// Position of the first query row.  It is in device memory, where no check of the host's sees it: below -sq no row
// sees a key and from skv on every row sees all of them, so the value is held between the two, and sums with
// row numbers stay small.
__device__ __forceinline__ int chunk_offset(const int32_t *chunk_start, int sq, int skv) {
  return chunk_start ? min(max(chunk_start[0], -sq), skv) : 0;
}

// The wavefronts of a workgroup are four consecutive (row block of 32 rows, query head) pairs of a head group, row block by row block:
// groups of four heads where a KV head has a multiple of four (a workgroup is four heads of one row block), all heads of it otherwise
// (two heads: two row blocks; five: the heads of one row block and part of the next).  One head per workgroup where their number is no
// multiple of two left three of four wavefronts without rows in a chunk of 32 and read K and V once per head.
__device__ __forceinline__ int row_blocks(const PrefillArgs &a) { return (a.sq + kRowsPerWave - 1) / kRowsPerWave; }
// Row block of the last pair of workgroup `wg` of a head group.
__device__ __forceinline__ int last_row_block(const PrefillArgs &a, int wg) {
  return min(quotient(a.by_head_group, 4 * wg + 3), row_blocks(a) - 1);
}

// Head group y and rank (0: the last row blocks, heavy ones first) of attention workgroup wg.  Workgroups are dealt to the 8 XCDs
// round-robin by linear id, and each XCD has its own L2: all workgroups of a group run on one XCD, one after the other, so that its
// K / V is fetched by one L2 only and stays resident there.  The groups left over when the rounds of eight are dealt are spread over all
// XCDs, one, two or four to each where they are a power of two: on an XCD each they left the others idle (two groups, one prompt of 4096 tokens with
// 8 / 2 heads of 64: 80 -> 51 us; 1312 rows behind 9152 128 -> 51).  `spread` (spreads_groups in prefill_parts.h) deals all groups
// over all XCDs, the workgroups of one after the other's, so that few of an XCD's are of one group.
__host__ __device__ __forceinline__ bool workgroup_place(const PrefillArgs &a, int wg, int &y, int &rank) {
  const int t = wg - a.full_rounds * 8 * a.spg;
  if (t < 0) {
    const int slot = wg >> 3, round = quotient(a.by_spg, slot);
    y = round * 8 + (wg & 7), rank = slot - round * a.spg;
    return true;
  }
  if (a.rest == 0) return false;
  const int q = quotient(a.by_rest, t), r = t - q * a.by_rest.d;
  rank = a.spread ? r : q;
  y = a.full_rounds * 8 + (a.spread ? q : r);
  return q < (a.spread ? a.rest : a.spg);
}
// ... and the host's side: the fields it reads, for `heads` query heads per head group and `spg` workgroups per group (0: as many as there are row
// blocks); the grid, a multiple of 8.
inline int lay_out(PrefillArgs &a, int heads, int spg = 0, bool spread = false) {
  const int groups = a.batch * (a.hq / heads);
  const int pairs = (a.sq + kRowsPerWave - 1) / kRowsPerWave * heads;
  a.head_group = heads, a.by_head_group = divisor(heads);
  a.spg = spg > 0 ? spg : (pairs + 3) / 4;
  a.spread = spread, a.full_rounds = spread ? 0 : groups / 8, a.rest = spread ? groups : groups % 8;
  a.by_spg = divisor(a.spg), a.by_rest = divisor(spread ? a.spg : std::max(a.rest, 1));
  a.by_groups = divisor(a.hq / heads), a.by_group_heads = divisor(a.hq / a.hkv);
  return a.full_rounds * 8 * a.spg + (a.rest * a.spg + 7) / 8 * 8;
}

// LDS geometry of one stage: the K tile (64 rows of D elements) followed by the V tile.
// Chunk c (16 bytes) of row r is stored at chunk position c ^ swz(r).
//   K fragments are read by 16 lanes of consecutive rows at one logical chunk: the 16
//   positions must differ (rows of >= 256 bytes) or, for 128-byte rows, differ within each
//   pair of rows that shares a 256-byte bank line.
//   V fragments are read, per 32 lanes, as 4 consecutive rows x 4 consecutive chunks.
template <int D>
struct Tile {
  static constexpr int RB = 2 * D;                 // row bytes
  static constexpr int CPR = D / 8;                // 16-byte chunks per row
  static constexpr int RPI = 1024 / RB;            // rows covered by one wavefront load
  static constexpr int NI = kKeysPerTile / RPI / 4;  // loads per wavefront per tile and tensor
  static constexpr int TILE_BYTES = kKeysPerTile * RB;
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES;
  __device__ static constexpr int swz_k(int r) { return RB >= 256 ? (r & 15) : ((r >> 1) & 7); }
  __device__ static constexpr int swz_v(int r) { return RB >= 256 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); }
};

// The cache fill that rides along with a dense prefill: workgroup f (counted from the end of
// the attention workgroups) copies fill_rows_per_wg(D) token rows (128 KiB, 64 at head size 64) of one (tensor, batch entry, KV head)
// from the dense K / V operand into the paged cache, with the semantics of the fill operator
// (rows whose table row or block is out of range are skipped).  Pure memory work that runs in
// the shadow of the matrix-bound attention workgroups; nothing in this launch reads the caches.
// 16-byte loads in flight per thread (head size 64: what fits the registers of three workgroups per CU)
constexpr int fill_passes(int d) { return d == 64 ? 16 : 32; }
constexpr int fill_rows_per_wg(int d) { return fill_passes(d) * (256 / (d / 8)); }

template <int D>
__device__ __forceinline__ void fill_workgroup(const PrefillArgs &a, int f) {
  constexpr int CPR = D / 8;        // 16-byte chunks per row
  constexpr int RPP = 256 / CPR;    // rows per pass of the 256 threads
  constexpr int NP = fill_passes(D);
  constexpr int kFillRows = fill_rows_per_wg(D);
  const int chunks = (a.skv + kFillRows - 1) / kFillRows;
  const int c0 = f % chunks;
  int r = f / chunks;
  const int h = r % a.hkv;
  r /= a.hkv;
  const int b = r % a.batch;
  const bool is_v = r / a.batch != 0;
  int64_t row = a.fill_bidx ? load_index(a.fill_bidx, a.fill_bidx_i64, b) : 0;
  if (row < 0 || row >= a.fill_rows) return;
  const uint16_t *src = (is_v ? a.v : a.k) + b * a.kv_bs + h * a.kv_hs;
  uint16_t *cache = is_v ? a.fill_vc : a.fill_kc;
  const int32_t *pt = a.fill_pt + row * a.fill_pt_rs;
  const int t0 = c0 * kFillRows + (int)threadIdx.x / CPR, c = (int)threadIdx.x % CPR;
  // every load (rows and table entries) is requested before the first store: the compiler
  // cannot move a load across a store that might alias it, and a table entry per pass would
  // otherwise cost a round trip each
  // A prompt of a quarter of the passes takes no more: 30 of 32 were the last row of 32 tokens again, and a fifth of a short launch that has more
  // workgroups than there are CUs (16 / 16 heads of 128, 5 x 32 tokens 5.8 -> 4.9 us, 8 x 32 5.95 -> 5.0, 8 x 64 6.0 -> 5.7; 4 x 32, with a CU for each,
  // 4.9).  Not so for the rest of longer ones, whose attention workgroups start less well behind fills that end early: 7 x 256 13.0 / 13.2, 7 x 640
  // 35.0 / 35.3, 4 x 640 of 16 / 8 heads of 256 39.3 / 40.1; nor at 256, where a CU has one workgroup: 8 x 64 7.73 / 7.80.
  constexpr int NQ = NP / 4;
  const int quarters = D <= 128 && a.skv <= NQ * RPP ? 1 : 4;
  u32x4 val[NP];
  int phys[NP];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q >= quarters) break;
#pragma unroll
    for (int p = q * NQ; p < (q + 1) * NQ; ++p) {
      const int t = min(t0 + p * RPP, a.skv - 1);
      val[p] = *reinterpret_cast<const u32x4 *>(src + (int64_t)t * a.kv_ts + 8 * c);
      phys[p] = pt[div_block(a, t)];
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q >= quarters) break;
#pragma unroll
    for (int p = q * NQ; p < (q + 1) * NQ; ++p) {
      const int t = t0 + p * RPP;
      const int off = t - div_block(a, t) * a.bs;
      // (no exit inside: the arrays must stay in registers)
      if (t < a.skv && (unsigned)phys[p] < (unsigned)a.nb)
        __builtin_nontemporal_store(val[p], reinterpret_cast<u32x4 *>(cache + (((int64_t)phys[p] * a.hkv + h) * a.bs + off) * D + 8 * c));
    }
  }
}

// Index of this workgroup among the attention workgroups of a dense launch that may carry a fill;
// negative: it was a fill workgroup and is done.
template <int D>
__device__ __forceinline__ int attention_workgroup(const PrefillArgs &a, int wg) {
  if (a.fill_kc == nullptr) return wg;
  const int per = 8 * (a.attn_per_fill + 1);
  const int sg = wg / per, m = wg - sg * per;
  if (sg >= a.fill_groups) return wg - 8 * a.fill_groups;
  if (m < 8 * a.attn_per_fill) return sg * 8 * a.attn_per_fill + m;
  const int f = sg * 8 + (m - 8 * a.attn_per_fill);
  if (f < a.n_fill) fill_workgroup<D>(a, f);
  return -1;
}

// The grid of a dense launch with a fill, from its attention workgroups (a multiple of 8): the fill
// workgroups are spread over the launch in groups of 8, one group behind every attn_per_fill groups
// of attention workgroups, so that their memory traffic runs while the neighbouring workgroups keep
// the matrix pipes busy (all of them at the end of the launch cost as much as two separate fills).
inline int grid_with_fill(PrefillArgs &b, int grid, int d) {
  b.n_fill = 2 * b.batch * b.hkv * ((b.skv + fill_rows_per_wg(d) - 1) / fill_rows_per_wg(d));
  const int fg = (b.n_fill + 7) / 8, ag = grid / 8;
  b.fill_groups = fg;
  b.attn_per_fill = ag >= fg ? ag / fg : 1;
  // fewer attention groups than fill groups: one of each per super-group, and the attention
  // slots past the last real one exit at once (the kernels' range check)
  return ag >= fg ? grid + 8 * fg : 16 * fg;
}

// prefill_stream.hip: whether the streaming kernel serves this launch, and the launch.
bool stream_serves(const PrefillArgs &a, int head_size);
// Whether a pass over block-float-8 caches, with `room` bytes of scratch, is worth expanding into bfloat16 copies for it.
bool stream_expands(const PrefillArgs &a, int head_size, int64_t room);
// Bytes of scratch with which it splits the launch over the keys (0: it would not); stream_serves launches only.
int64_t stream_part_bytes(const PrefillArgs &a, int head_size);
int launch_stream(const PrefillArgs &a, int head_size, hipStream_t st);
int launch_stream_d64(const PrefillArgs &a, hipStream_t st);
int launch_stream_d256(const PrefillArgs &a, hipStream_t st);
// The streaming kernel for keys of 128 + 64 features (dense, causal or not, kv length a multiple of 32).
int launch_stream_wide(const PrefillArgs &a, hipStream_t st);

}  // namespace ttpa
