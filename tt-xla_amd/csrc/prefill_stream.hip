// Streaming prefill attention for gfx950: head size 128, no explicit mask, K / V readable in whole
// blocks of 32 keys (dense, or paged with a block size that is a multiple of 32).  The matrix pipe bounds it:
// 16 v_mfma_f32_32x32x16_bf16 per block of 32 keys and wavefront, with the vector work of the softmax
// between them.
//
// The work split is that of prefill.hip (four wavefronts of 32 query rows share K / V in LDS: HPW
// heads of one KV head times 4 / HPW row blocks; all row blocks of a (batch entry, head group) on one
// XCD, heavy ones first).  The whole life of a workgroup behind its address set-up is one block of
// assembly, written by gen_prefill_stream.py, which documents the schedule and the state on entry.
// Against the compiler-scheduled loop of prefill.hip on the same shapes (a whole pass): window of 1024
// keys, 2 x 4096 tokens, 32 / 8 heads 160 -> 137 us; 4 x 2048 tokens, 16 / 16 heads 118 -> 98 us and 16 / 8
// heads 99 -> 83 us; 2 x 2048 tokens, 40 / 8 heads 126 -> 103 us; 2 x 512-token chunks behind 4096 tokens,
// 16 / 16 heads 103 -> 81 us.
//
// A launch of few row blocks over many keys (the chunk of one request far into its sequence: 128
// workgroups for 512 rows of 32 / 8 heads, on 256 CUs that hold two each) is split over the keys:
// several workgroups per row block, each with a share of the 32-key blocks, hand float accumulators
// to prefill_merge_kernel.  512 rows behind 8192 tokens: blocks of 64 139 -> 80 us for the pass, blocks of 32
// 231 -> 81 us (unsplit on the plain loop before); 256 rows of 16 / 16 heads behind 8192 228 -> 67 us.  Blocks
// of 32 alone, where nothing is split: 4 x 512 rows behind 4096 tokens 180 -> 144 us.
#include "prefill_parts.h"
#include "build/prefill_stream_asm.h"

#include <algorithm>
#include <cstdlib>

namespace ttpa {
namespace {

constexpr int kD = 128;

// kPaged: cache blocks of whole 64-key tiles (two 32-key blocks share a table entry); kPaged32: of whole
// 32-key blocks (an entry per block costs scalar instructions in every iteration, not in every other one)
// kDenseWide: keys of 128 + 64 features (the latent layers' prompts with K and V expanded per head): 20 matrix
// instructions per block of 32 keys; 4 x 2048 tokens, 16 heads: 8.6e10 flop in 100 us, where the absorbed form's
// 2.9e11 took 281
enum StreamForm { kDense = 0, kDenseWindow = 1, kPaged = 2, kPaged32 = 3, kDenseWide = 4 };

// The assembly is bound to the registers its text names through constraint strings; everything else it
// touches is on the clobber list.  The requests of a workgroup's first blocks are a block of assembly of their own, issued in front
// of the Q loads so that the two round trips to memory overlap.  (Scalars only: with the per-lane
// offsets in the same struct the compiler keeps the whole of it in vector registers.)
struct StreamRequests {
  uint64_t kbase, vbase;       // dense: the first block of K / V; paged: the caches (both minus 1024 bytes)
  uint32_t stride;             // dense: bytes from a 32-key block to the next; paged: bytes of a (cache block, head) slab
  uint32_t m0_base;            // LDS address of the wavefront's first segment in K slot 0
  int k_requests, v_requests;  // blocks not requested yet
  uint64_t off0, off1, off2;   // paged: byte offsets of tiles 0, 1, 2 in a cache
};

__device__ __forceinline__ void stream_first_dense(StreamRequests &r, const u32x2 &ldk, const u32x2 &ldv) {
  asm volatile(TTPA_STREAM_FIRST_TEXT_DENSE
               : "+{s[64:65]}"(r.kbase), "+{s[66:67]}"(r.vbase), "+{s71}"(r.k_requests), "+{s73}"(r.v_requests)
               : "{v[188:189]}"(ldk), "{v[190:191]}"(ldv), "{s68}"(r.stride), "{s72}"(r.m0_base)
               : "memory", "scc", "m0");
}

__device__ __forceinline__ void stream_first_paged(StreamRequests &r, const u32x2 &ldk, const u32x2 &ldv) {
  asm volatile(TTPA_STREAM_FIRST_TEXT_PAGED
               : "+{s71}"(r.k_requests), "+{s73}"(r.v_requests)
               : "{v[188:189]}"(ldk), "{v[190:191]}"(ldv), "{s[64:65]}"(r.kbase), "{s[66:67]}"(r.vbase),
                 "{s72}"(r.m0_base), "{s[84:85]}"(r.off1), "{s[86:87]}"(r.off2), "{s[98:99]}"(r.off0)
               : "memory", "scc", "m0", "s90", "s91");
}

// Values the compiler may hold in vector registers although they are the same in every lane: the
// block binds them to scalar registers.
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint32_t uni(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
__device__ __forceinline__ uint64_t uni(uint64_t x) {
  return address_from_words(__builtin_amdgcn_readfirstlane((int)(uint32_t)x), __builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32)));
}

__device__ __forceinline__ void stream_first_paged32(StreamRequests &r, const u32x2 &ldk, const u32x2 &ldv, const uint64_t (&off)[5]) {
  asm volatile(TTPA_STREAM_FIRST_TEXT_PAGED32
               : "+{s71}"(r.k_requests), "+{s73}"(r.v_requests)
               : "{v[188:189]}"(ldk), "{v[190:191]}"(ldv), "{s[64:65]}"(r.kbase), "{s[66:67]}"(r.vbase),
                 "{s72}"(r.m0_base), "{s[50:51]}"(off[0]), "{s[52:53]}"(off[1]), "{s[58:59]}"(off[2]), "{s[84:85]}"(off[3]),
                 "{s[98:99]}"(off[4])
               : "memory", "scc", "m0", "s90", "s91");
}

// The second part of the keys: its first block, bytes from a block to the next, the LDS address of the
// wavefront's segment, V's bytes per block, the lane's offset inside a block.
struct StreamWide {
  uint64_t base;
  uint32_t stride, m0, v_stride;
};

__device__ __forceinline__ void stream_first_wide(StreamRequests &r, StreamWide &w, const u32x2 &ldk, const u32x2 &ldv, uint32_t ldp) {
  asm volatile(TTPA_STREAM_FIRST_TEXT_DENSE_WIDE
               : "+{s[64:65]}"(r.kbase), "+{s[66:67]}"(r.vbase), "+{s[30:31]}"(w.base), "+{s71}"(r.k_requests), "+{s73}"(r.v_requests)
               : "{v[188:189]}"(ldk), "{v[190:191]}"(ldv), "{v248}"(ldp), "{s68}"(r.stride), "{s72}"(r.m0_base),
                 "{s32}"(w.stride), "{s33}"(w.m0), "{s35}"(w.v_stride)
               : "memory", "scc", "m0");
}

// What a workgroup works on (see gen_prefill_stream.py): which row blocks, and what the block of
// assembly needs to set one up.
struct StreamItems {
  int k, j, spg, nqt;          // item counter (starts at 0), the workgroup's slot, slots, row blocks
  int sq, skv, offset, causal;
  uint32_t q_row_bytes, out_row_bytes;
  int row0;                    // first query row of item 0
  int key0;                    // first key of its first block
};

#define TTPA_STREAM_COMMON_OUT                                                                        \
  "+{v[64:79]}"(q_lo), "+{v[80:95]}"(q_hi), "+{s[64:65]}"(r.kbase), "+{s[66:67]}"(r.vbase), "+{s70}"(nblk), \
      "+{s71}"(r.k_requests), "+{s73}"(r.v_requests), "+{s40}"(it.k), "+{s57}"(it.row0), "+{s75}"(it.key0)
#define TTPA_STREAM_COMMON_IN                                                                       \
  "{v[176:183]}"(koff), "{v[184:187]}"(voff), "{v[188:189]}"(ldk), "{v[190:191]}"(ldv),         \
      "{v[216:217]}"(q_base), "{v[218:219]}"(out_base), "{v220}"(lane_n), "{v221}"(lane_h4),       \
      "{s68}"(r.stride), "{s69}"(c), "{s72}"(r.m0_base), "{s41}"(it.j), "{s42}"(it.spg), "{s43}"(it.nqt), \
      "{s44}"(it.sq), "{s45}"(it.skv), "{s46}"(it.offset), "{s47}"(it.causal), "{s48}"(it.q_row_bytes),  \
      "{s49}"(it.out_row_bytes)

// Everything behind the first requests of item 0, through the stored output rows of the last item.
// q_lo / q_hi: the eight Q fragments of item 0; koff / voff: the lane's LDS addresses of its K and
// V^T fragments in slot 0 of the K and V rings; nblk: the 32-key blocks of item 0; kbase0 / vbase0:
// block 0 of K / V again, for the items that follow.
__device__ __forceinline__ void stream_items_dense(StreamRequests &r, StreamItems &it, u32x16 q_lo, u32x16 q_hi,
                                                   const u32x8 &koff, const u32x4 &voff, const u32x2 &ldk,
                                                   const u32x2 &ldv, uint64_t q_base, uint64_t out_base, int lane_n,
                                                   int lane_h4, float c, int nblk, uint64_t kbase0, uint64_t vbase0) {
  asm volatile(TTPA_STREAM_LOOP_TEXT_DENSE
               : TTPA_STREAM_COMMON_OUT
               : TTPA_STREAM_COMMON_IN, "{s[50:51]}"(kbase0), "{s[52:53]}"(vbase0)
               : "memory", "vcc", "scc", "m0", "v208", "v209", TTPA_STREAM_LOOP_CLOBBERS);
}

// Dense with a sliding window: lowest is the first key of the lane's row minus 4 (lane / 32), low_to the
// key from which on no row of the wavefront needs a mask from below.
__device__ __forceinline__ void stream_items_window(StreamRequests &r, StreamItems &it, u32x16 q_lo, u32x16 q_hi,
                                                    const u32x8 &koff, const u32x4 &voff, const u32x2 &ldk,
                                                    const u32x2 &ldv, uint64_t q_base, uint64_t out_base, int lane_n,
                                                    int lane_h4, float c, int nblk, int lowest, int low_to) {
  asm volatile(TTPA_STREAM_LOOP_TEXT_DENSE_WINDOW
               : TTPA_STREAM_COMMON_OUT
               : TTPA_STREAM_COMMON_IN, "{v209}"(lowest), "{s34}"(low_to)
               : "memory", "vcc", "scc", "m0", "v208", TTPA_STREAM_LOOP_CLOBBERS);
}

__device__ __forceinline__ void stream_items_wide(StreamRequests &r, StreamItems &it, StreamWide &w, u32x16 q_lo, u32x16 q_hi,
                                                  u32x16 q_second, const u32x8 &koff, const u32x4 &poff, const u32x4 &voff,
                                                  const u32x2 &ldk, const u32x2 &ldv, uint32_t ldp, uint64_t q_base, uint64_t out_base,
                                                  int lane_n, int lane_h4, float c, int nblk) {
  asm volatile(TTPA_STREAM_LOOP_TEXT_DENSE_WIDE
               : TTPA_STREAM_COMMON_OUT, "+{s[30:31]}"(w.base)
               : TTPA_STREAM_COMMON_IN, "{v[228:243]}"(q_second), "{v[244:247]}"(poff), "{v248}"(ldp), "{s32}"(w.stride),
                 "{s33}"(w.m0), "{s35}"(w.v_stride)
               : "memory", "vcc", "scc", "m0", "v208", TTPA_STREAM_LOOP_CLOBBERS);
}

// Where a workgroup that takes a part of the keys leaves its result (0: the whole result goes to the output).
struct StreamPart {
  uint64_t stats, acc;
};

// The block-table state of the paged forms: table entries per cache block, the raw entry (blocks of 32:
// the two raw entries) that follow the first requests, where they and the next requested one lie in their
// cache blocks, the address of the latter, and how many are left to request.
struct StreamTable {
  int kv_heads, kv_head, num_blocks, per_block;
  int entry, entry2;
  int read_in_block, request_in_block;
  uint64_t entry_ptr;
  int entry_requests;
};

__device__ __forceinline__ void stream_items_paged(StreamRequests &r, StreamItems &it, StreamTable &t, StreamPart &part,
                                                   u32x16 q_lo, u32x16 q_hi, const u32x8 &koff, const u32x4 &voff, const u32x2 &ldk,
                                                   const u32x2 &ldv, uint64_t q_base, uint64_t out_base, int lane_n,
                                                   int lane_h4, float c, int nblk) {
  const int read_in_block0 = t.read_in_block, request_in_block0 = t.request_in_block, entry0 = t.entry;
  const uint64_t entry_ptr0 = t.entry_ptr, off1 = r.off1, off2 = r.off2;
  asm volatile(TTPA_STREAM_LOOP_TEXT_PAGED
               : TTPA_STREAM_COMMON_OUT, "+{s80}"(t.read_in_block), "+{s81}"(t.request_in_block),
                 "+{s[82:83]}"(t.entry_ptr), "+{s[84:85]}"(r.off1), "+{s[86:87]}"(r.off2), "+{s96}"(t.entry_requests),
                 "+{v208}"(t.entry), "+{s[38:39]}"(part.acc)
               : TTPA_STREAM_COMMON_IN, "{s76}"(t.kv_heads), "{s77}"(t.kv_head), "{s78}"(t.num_blocks),
                 "{s79}"(t.per_block), "{s[98:99]}"(r.off0), "{s[50:51]}"(off1), "{s[52:53]}"(off2),
                 "{s54}"(entry0), "{s55}"(read_in_block0), "{s56}"(request_in_block0), "{s[58:59]}"(entry_ptr0),
                 "{s[36:37]}"(part.stats)
               : "memory", "vcc", "scc", "m0", TTPA_STREAM_LOOP_CLOBBERS);
}

__device__ __forceinline__ void stream_items_paged32(StreamRequests &r, StreamItems &it, StreamTable &t, StreamPart &part, uint64_t off3,
                                                     uint64_t off4, u32x16 q_lo, u32x16 q_hi, const u32x8 &koff, const u32x4 &voff,
                                                     const u32x2 &ldk, const u32x2 &ldv, uint64_t q_base, uint64_t out_base,
                                                     int lane_n, int lane_h4, float c, int nblk) {
  asm volatile(TTPA_STREAM_LOOP_TEXT_PAGED32
               : TTPA_STREAM_COMMON_OUT, "+{s80}"(t.read_in_block), "+{s81}"(t.request_in_block),
                 "+{s[82:83]}"(t.entry_ptr), "+{s[84:85]}"(off3), "+{s[98:99]}"(off4), "+{s96}"(t.entry_requests),
                 "+{v208}"(t.entry), "+{v211}"(t.entry2), "+{s[38:39]}"(part.acc)
               : TTPA_STREAM_COMMON_IN, "{s76}"(t.kv_heads), "{s77}"(t.kv_head), "{s78}"(t.num_blocks),
                 "{s79}"(t.per_block), "{s[36:37]}"(part.stats)
               : "memory", "vcc", "scc", "m0", "s86", "s87", TTPA_STREAM_LOOP_CLOBBERS);
}

template <int HPW, int FORM>
__global__ __launch_bounds__(256, 2) void prefill_stream_kernel(PrefillArgs a) {
  constexpr int RPW = 4 / HPW;  // row blocks per workgroup
  constexpr int D = kD;
  constexpr bool PAGED = FORM == kPaged || FORM == kPaged32, WIDE = FORM == kDenseWide;
  using T = Tile<D>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  int wg = blockIdx.x;
  if constexpr (!PAGED && !WIDE) {
    wg = attention_workgroup<D>(a, wg);
    if (wg < 0) return;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int nqt = (a.sq + kRowsPerWave * RPW - 1) / (kRowsPerWave * RPW);
  const int groups = a.hq / HPW;
  // The part is the slowest index: the workgroups of part 0, the only ones with work where the keys are few, are dealt over the
  // XCDs and CUs as in a launch that is not split.  (As the fastest index, they met on half of the CUs or a quarter: 256
  // workgroups over 512 keys 20.5 us, 16.3 this way.)
  const int part = PAGED ? blockIdx.y : 0;
  const int xcd = wg & 7, slot = wg >> 3;
  const int yl = slot / a.spg;
  const int y = yl * 8 + xcd;
  if (y >= a.batch * groups) return;  // grid is padded to a multiple of 8 groups
  const int item0 = slot - yl * a.spg;
  const int qt = nqt - 1 - item0;
  const int b = y / groups;
  const int hq0 = (y - b * groups) * HPW;
  const int hk = hq0 / (a.hq / a.hkv);
  const int hq = hq0 + wave % HPW;
  const int row0 = (qt * RPW + wave / HPW) * kRowsPerWave;  // first query row of the wavefront
  const int offset = a.causal ? chunk_offset(a.chunk_start, a.sq, a.skv) : 0;

  // keys the workgroup can see, in blocks of 32
  const int wg_last_row = min(a.sq, (qt + 1) * kRowsPerWave * RPW) - 1;
  const int kv_end = a.causal ? min(a.skv, offset + wg_last_row + 1) : a.skv;
  int first_block = FORM == kDenseWindow ? max(0, offset + qt * kRowsPerWave * RPW - a.window + 1) / kBlockKeys : 0;
  // (at least one: the loop counts blocks down to zero.  Where no row sees a key, a chunk that starts at a negative
  // position, block 0 is read and masked, and the rows come out as NaN, softmax over nothing)
  int nblk = __builtin_amdgcn_readfirstlane(max((kv_end + kBlockKeys - 1) / kBlockKeys - first_block, 1));
  bool whole = true;  // this workgroup sees all keys of its rows
  if constexpr (PAGED) {
    if (a.parts > 1) {
      const int share = __builtin_amdgcn_readfirstlane(blocks_per_part(a, offset));
      whole = share >= nblk;
      first_block = part * share;
      nblk = min(share, nblk - first_block);
      if (nblk <= 0) return;
    }
  }

  int spg = a.spg;
  if (a.spg_even > 0) {
    const int lightest = a.causal ? min(offset + kRowsPerWave, a.skv) : a.skv;
    const int heaviest = a.causal ? min(offset + a.sq, a.skv) : a.skv;
    if (4 * lightest >= 3 * heaviest) {
      spg = a.spg_even;
      if (item0 >= spg) return;
    }
  }

  // ---- first requests, in front of the Q loads ----------------------------------------------------
  StreamRequests sreq;
  u32x2 ldk, ldv;
  const uint32_t lds0 = lds_address(smem);
  const uint32_t row_bytes = PAGED ? (uint32_t)T::RB : 2u * (uint32_t)a.kv_ts;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    // a block is 8 segments of 1 KiB; wavefront w requests segments 2 w and 2 w + 1
    const int r = (2 * wave + j) * T::RPI + lane / T::CPR, cp = lane % T::CPR;
    ldk[j] = (uint32_t)r * row_bytes + 16u * (uint32_t)(cp ^ T::swz_k(r)) + 1024u - 1024u * j;
    ldv[j] = (uint32_t)r * (WIDE ? 2u * (uint32_t)a.v_ts : row_bytes) + 16u * (uint32_t)(cp ^ T::swz_v(r)) + 1024u - 1024u * j;
  }
  StreamWide wide;
  uint32_t ldp = 0;
  if constexpr (WIDE) {
    // a block of the second part is 4 segments of eight 128-byte rows, one per wavefront
    const int r = 8 * wave + (lane >> 3);
    ldp = (uint32_t)r * 2u * (uint32_t)a.k2_ts + 16u * (uint32_t)((lane & 7) ^ Tile<64>::swz_k(r));
    wide.base = uni(reinterpret_cast<uint64_t>(a.k2 + b * a.k2_bs + hk * a.k2_hs));
    wide.stride = (uint32_t)(2 * kBlockKeys * a.k2_ts), wide.v_stride = (uint32_t)(2 * kBlockKeys * a.v_ts);
    wide.m0 = uni(lds0 + TTPA_STREAM_WIDE_P_RING + 1024u * (uint32_t)wave);
  }
  sreq.m0_base = uni(lds0 + 2048u * (uint32_t)wave);
  sreq.k_requests = sreq.v_requests = nblk;
  sreq.off0 = sreq.off1 = sreq.off2 = 0;
  StreamTable tab;
  StreamPart out_part = {0, 0};
  uint64_t off[5];
  uint64_t kbase0 = 0, vbase0 = 0;
  if constexpr (!PAGED) {
    const int64_t head = b * a.kv_bs + hk * a.kv_hs + (int64_t)first_block * kBlockKeys * a.kv_ts;
    kbase0 = uni(reinterpret_cast<uint64_t>(a.k + head) - 1024u);
    vbase0 = uni(reinterpret_cast<uint64_t>(a.v + (WIDE ? b * a.v_bs + hk * a.v_hs : head)) - 1024u);
    sreq.kbase = kbase0, sreq.vbase = vbase0;
    sreq.stride = (uint32_t)(2 * kBlockKeys * a.kv_ts);
    if constexpr (WIDE) stream_first_wide(sreq, wide, ldk, ldv, ldp);
    else stream_first_dense(sreq, ldk, ldv);
  } else {
    // keys that share a table entry are a multiple of a unit (a 64-key tile, a 32-key block); the first FIRST
    // units are requested here, the loop takes raw entries from there on
    constexpr int UNIT = FORM == kPaged ? kKeysPerTile : kBlockKeys;
    constexpr int FIRST = FORM == kPaged ? 3 : 5, RAW = FORM == kPaged ? 1 : 2;
    const int per = a.bs / UNIT, last = a.w * per - 1;  // (entries exist for every unit of the table)
    const int unit0 = first_block * kBlockKeys / UNIT;
    sreq.kbase = reinterpret_cast<uint64_t>(a.k) - 1024u;
    sreq.vbase = reinterpret_cast<uint64_t>(a.v) - 1024u;
    sreq.stride = (uint32_t)a.bs * (uint32_t)T::RB;
    int raw[FIRST + RAW];
#pragma unroll
    for (int t = 0; t < FIRST + RAW; ++t) raw[t] = a.pt[(int64_t)b * a.pt_rs + min(unit0 + t, last) / per];
#pragma unroll
    for (int t = 0; t < FIRST; ++t) {
      int phys = __builtin_amdgcn_readfirstlane(raw[t]);
      if ((unsigned)phys >= (unsigned)a.nb) phys = 0;
      off[t] = uni((uint64_t)((int64_t)phys * a.hkv + hk) * sreq.stride + (uint64_t)(min(unit0 + t, last) % per) * (UNIT * T::RB));
    }
    tab.kv_heads = uni(a.hkv), tab.kv_head = uni(hk), tab.num_blocks = uni(a.nb), tab.per_block = uni(per);
    tab.entry = raw[FIRST], tab.entry2 = raw[FIRST + RAW - 1];
    const int next = unit0 + FIRST;
    tab.read_in_block = uni(next % per), tab.request_in_block = uni((next + RAW) % per);
    tab.entry_ptr = uni(reinterpret_cast<uint64_t>(a.pt + (int64_t)b * a.pt_rs + (next + RAW) / per));
    tab.entry_requests = uni(max((nblk - 1) / (UNIT / kBlockKeys) + 1 - FIRST - RAW, 0));
    if constexpr (FORM == kPaged) {
      sreq.off0 = off[0], sreq.off1 = off[1], sreq.off2 = off[2];
      stream_first_paged(sreq, ldk, ldv);
    } else {
      stream_first_paged32(sreq, ldk, ldv, off);
    }
    if (!whole) {
      const PartLayout lay = part_layout(a, kRowsPerWave * RPW);
      const int64_t at = (((int64_t)part * a.batch + b) * a.hq + hq) * lay.row_blocks + qt * RPW + wave / HPW;
      out_part.acc = uni(reinterpret_cast<uint64_t>(a.part_acc + at * part_acc_floats(D)));
      out_part.stats = uni(reinterpret_cast<uint64_t>(a.part_acc + lay.slots * part_acc_floats(D) + at * (2 * kRowsPerWave)));
    }
  }
  // Q fragments behind the requests (B operand: lane n = query row, 8 head-dim elements per k-step)
  u32x16 q_lo, q_hi;
  {
    const int qrow = min(row0 + n, a.sq - 1);
    const uint16_t *qp = a.q + b * a.q_bs + hq * a.q_hs + (int64_t)qrow * a.q_ts + 8 * h;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint4 lo = *reinterpret_cast<const uint4 *>(qp + 16 * s), hi = *reinterpret_cast<const uint4 *>(qp + 16 * (s + 4));
      q_lo[4 * s] = lo.x, q_lo[4 * s + 1] = lo.y, q_lo[4 * s + 2] = lo.z, q_lo[4 * s + 3] = lo.w;
      q_hi[4 * s] = hi.x, q_hi[4 * s + 1] = hi.y, q_hi[4 * s + 2] = hi.z, q_hi[4 * s + 3] = hi.w;
    }
  }
  u32x16 q_second;
  u32x4 po;
  if constexpr (WIDE) {
    const uint16_t *qp = a.q2 + b * a.q2_bs + hq * a.q2_hs + (int64_t)min(row0 + n, a.sq - 1) * a.q2_ts + 8 * h;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint4 x = *reinterpret_cast<const uint4 *>(qp + 16 * s);
      q_second[4 * s] = x.x, q_second[4 * s + 1] = x.y, q_second[4 * s + 2] = x.z, q_second[4 * s + 3] = x.w;
      po[s] = lds0 + TTPA_STREAM_WIDE_P_RING + (uint32_t)(n * 128 + 16 * ((2 * s + h) ^ Tile<64>::swz_k(n)));
    }
  }
  // LDS operand addresses of the lane inside slot 0 of the K ring and of the V ring: K fragment of k-step
  // s, V^T fragment of output block db (through the transposing LDS load; the layout of prefill.hip)
  u32x8 ko;
#pragma unroll
  for (int s = 0; s < 8; ++s) ko[s] = lds0 + (uint32_t)(n * T::RB + 16 * ((2 * s + h) ^ T::swz_k(n)));
  u32x4 vo;
  {
    const int grp = lane >> 4, a16 = lane & 15, vr = 4 * (grp >> 1) + (a16 >> 2);
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const int c = 4 * db + 2 * (grp & 1) + ((a16 & 3) >> 1);
      vo[db] = lds0 + (WIDE ? TTPA_STREAM_WIDE_V_RING : TTPA_STREAM_V_RING) + (uint32_t)(vr * T::RB + 16 * (c ^ T::swz_v(vr)) + 8 * (a16 & 1));
    }
  }
  StreamItems it;
  it.k = 0, it.j = uni(item0), it.spg = uni(spg), it.nqt = uni(nqt);
  it.sq = uni(a.sq), it.skv = uni(a.skv), it.offset = uni(offset), it.causal = uni(a.causal);
  it.q_row_bytes = uni(2u * (uint32_t)a.q_ts), it.out_row_bytes = uni(2u * (uint32_t)a.out_ts);
  it.row0 = __builtin_amdgcn_readfirstlane(row0);
  it.key0 = uni(first_block * kBlockKeys);
  // per lane: row 0 of the lane's head, at the lane's 8 (lane / 32) / 4 (lane / 32) elements
  const uint64_t q_base = reinterpret_cast<uint64_t>(a.q + b * a.q_bs + hq * a.q_hs + 8 * h);
  const uint64_t out_base = reinterpret_cast<uint64_t>(a.out + b * a.out_bs + hq * a.out_hs + 8 * h);
  if constexpr (FORM == kDense) {
    stream_items_dense(sreq, it, q_lo, q_hi, ko, vo, ldk, ldv, q_base, out_base, n, 4 * h, a.scale_log2e, nblk, kbase0, vbase0);
  } else if constexpr (FORM == kDenseWindow) {
    const int lowest = offset + min(row0 + n, a.sq - 1) - a.window + 1 - 4 * h;
    const int low_to = uni(offset + row0 + kRowsPerWave - a.window);
    stream_items_window(sreq, it, q_lo, q_hi, ko, vo, ldk, ldv, q_base, out_base, n, 4 * h, a.scale_log2e, nblk, lowest, low_to);
  } else if constexpr (WIDE) {
    stream_items_wide(sreq, it, wide, q_lo, q_hi, q_second, ko, po, vo, ldk, ldv, ldp, q_base, out_base, n, 4 * h, a.scale_log2e, nblk);
  } else if constexpr (FORM == kPaged) {
    stream_items_paged(sreq, it, tab, out_part, q_lo, q_hi, ko, vo, ldk, ldv, q_base, out_base, n, 4 * h, a.scale_log2e, nblk);
  } else {
    stream_items_paged32(sreq, it, tab, out_part, off[3], off[4], q_lo, q_hi, ko, vo, ldk, ldv, q_base, out_base, n, 4 * h, a.scale_log2e, nblk);
  }
}

template <int HPW, int FORM>
int launch_form(const PrefillArgs &a, hipStream_t st) {
  constexpr int RPW = 4 / HPW;
  const int nqt = (a.sq + kRowsPerWave * RPW - 1) / (kRowsPerWave * RPW);
  static std::atomic<uint64_t> lds_ready{0};
  if (!ensure_dynamic_lds(reinterpret_cast<const void *>(&prefill_stream_kernel<HPW, FORM>), TTPA_STREAM_LDS_BYTES, lds_ready))
    return fail(TTPA_ERR_LAUNCH, "prefill: cannot reserve %d bytes of LDS", TTPA_STREAM_LDS_BYTES);
  const int ny8 = (a.batch * (a.hq / HPW) + 7) / 8;
  PrefillArgs b = a;
  // One workgroup per row block and head group, heavy blocks first, and the dispatcher deals them to the CUs
  // as slots free up: the loop can also give a workgroup several row blocks (spg workgroups per group,
  // TTPA_PREFILL_WGS_PER_GROUP), but one round of two workgroups per CU measured 204 us against 150 on
  // the 4 x 2048-token causal workload (a change of row block costs a workgroup about 4 us in which
  // nothing of its own overlaps, and a static deal cannot make up for workgroups that start late).
  b.spg = nqt, b.spg_even = 0;
  b.parts = 1;
  constexpr bool PAGED = FORM == kPaged || FORM == kPaged32;
  // (read on every call) an experiment's override: several row blocks per workgroup, each over all of its keys
  const char *e = HPW == 4 && (FORM == kDense || FORM == kPaged) ? getenv("TTPA_PREFILL_WGS_PER_GROUP") : nullptr;
  const int per_group = e ? atoi(e) : 0;
  if (PAGED && per_group <= 0 && a.part_acc && a.part_bytes >= part_bytes(a, HPW, kStreamSplit, kD)) set_parts(b, HPW, kStreamSplit);
  if (per_group > 0) {
    b.spg = std::min(nqt, per_group);
  } else if (HPW == 4 && (FORM == kDense || FORM == kPaged) && b.parts == 1) {
    // Row blocks of nearly one weight (a chunk far into its sequence, or no causal mask) that fill the
    // chip more than once: one round of workgroups with equal shares instead, which saves the later
    // rounds' start-up (267 -> 261 us on 4 x 512-token chunks behind 4096 tokens, 64 heads).  The
    // chunk's start is in device memory, so the kernel decides: the workgroups past the round exit.
    int cus = device_cus();
    if (cus <= 0) cus = 256;
    const int one_round = (2 * cus + ny8 * 8 - 1) / (ny8 * 8);
    b.spg_even = one_round < nqt && nqt % one_round == 0 ? one_round : 0;
  }
  int grid = b.spg * ny8 * 8;
  if (!PAGED && FORM != kDenseWide && a.fill_kc) grid = grid_with_fill(b, grid, kD);
  launch_dominant(&prefill_stream_kernel<HPW, FORM>, dim3(grid, b.parts), dim3(256), (size_t)TTPA_STREAM_LDS_BYTES, st, b);
  if (const int rc = check_launch("sdpa_prefill")) return rc;
  if (b.parts > 1) {
    prefill_merge_kernel<kD, RPW><<<dim3((b.sq + kRowsPerWave - 1) / kRowsPerWave, b.hq, b.batch), dim3(2 * kD), 0, st>>>(b);
    return check_launch("sdpa_prefill (merge of the parts)");
  }
  return TTPA_OK;
}

template <int HPW>
int launch_heads(const PrefillArgs &a, hipStream_t st) {
  if (a.pt) return a.bs % kKeysPerTile == 0 ? launch_form<HPW, kPaged>(a, st) : launch_form<HPW, kPaged32>(a, st);
  return a.window > 0 ? launch_form<HPW, kDenseWindow>(a, st) : launch_form<HPW, kDense>(a, st);
}

}  // namespace

// The line lies where the loop's unit does: whole blocks of 32 keys that lie in one piece, at the one head
// size whose register map is built.  A dense K / V that ends inside a block, smaller cache blocks,
// windows over a paged cache and explicit masks are the plain loop's.  Wherever both run, this one is
// faster (above) or, on passes of a few microseconds, equal.
bool stream_serves(const PrefillArgs &a, int head_size) {
  if (!a.stream || head_size != kD || a.mask != nullptr) return false;
  if (a.pt) return a.bs % kBlockKeys == 0 && a.window == 0;
  return a.skv % kBlockKeys == 0;
}

int64_t stream_part_bytes(const PrefillArgs &a, int head_size) {
  return a.pt && stream_serves(a, head_size) ? part_bytes(a, heads_per_workgroup(a), kStreamSplit, kD) : 0;
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
bool stream_expands(const PrefillArgs &a, int head_size, int64_t room) {
  if (!stream_serves(a, head_size)) return false;
  const int hpw = heads_per_workgroup(a), rows = kRowsPerWave * 4 / hpw;
  const int64_t row_blocks = (a.sq + rows - 1) / rows, readers = row_blocks * (a.hq / hpw / a.hkv);
  const int64_t parts = plain_part_bytes(a, kD, true);
  const bool splits = parts > 0 && parts <= room;
  // (a table has room for more keys than the chunk's: 8192 rows of it)
  const bool few = a.batch * a.keys_bound * a.hkv <= (a.keys_known ? 5120 : 8192);
  const bool pays = (row_blocks > 1 && (readers > 2 || a.keys_bound >= 512)) || few || part_bytes(a, hpw, kStreamSplit, kD) > 0 || (readers > (splits ? 3 : 2) && a.keys_bound >= 512);
  return pays && !(splits && readers <= 2);
}

int launch_stream_wide(const PrefillArgs &a, hipStream_t st) {
  switch (heads_per_workgroup(a)) {
    case 4: return launch_form<4, kDenseWide>(a, st);
    case 2: return launch_form<2, kDenseWide>(a, st);
    default: return launch_form<1, kDenseWide>(a, st);
  }
}

int launch_stream(const PrefillArgs &a, hipStream_t st) {
  switch (heads_per_workgroup(a)) {
    case 4: return launch_heads<4>(a, st);
    case 2: return launch_heads<2>(a, st);
    default: return launch_heads<1>(a, st);
  }
}

}  // namespace ttpa
