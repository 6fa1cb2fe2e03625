// Streaming prefill attention for gfx950: head size 128, no explicit mask, K / V readable in whole
// blocks of 32 keys (dense, or paged with a block size that is a multiple of 64).  The matrix pipe bounds it:
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
#include "prefill_common.h"
#include "build/prefill_stream_asm.h"

#include <algorithm>
#include <cstdlib>

namespace ttpa {
namespace {

constexpr int kD = 128;
constexpr int kBlockKeys = 32;

enum StreamForm { kDense = 0, kDenseWindow = 1, kPaged = 2 };

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

// Paged: entry is the raw table entry of tile 3, entry_ptr the address of tile 4's.
__device__ __forceinline__ void stream_items_paged(StreamRequests &r, StreamItems &it, u32x16 q_lo, u32x16 q_hi,
                                                   const u32x8 &koff, const u32x4 &voff, const u32x2 &ldk,
                                                   const u32x2 &ldv, uint64_t q_base, uint64_t out_base, int lane_n,
                                                   int lane_h4, float c, int nblk, int kv_heads, int kv_head, int num_blocks, int tiles_per_block,
                                                   int entry, uint64_t entry_ptr) {
  int read_in_block = 3 % tiles_per_block, request_in_block = 4 % tiles_per_block;
  const int read_in_block0 = read_in_block, request_in_block0 = request_in_block, entry0 = entry;
  const uint64_t entry_ptr0 = entry_ptr, off1 = r.off1, off2 = r.off2;
  int entry_requests = max((nblk - 1) / 2 - 3, 0);
  asm volatile(TTPA_STREAM_LOOP_TEXT_PAGED
               : TTPA_STREAM_COMMON_OUT, "+{s80}"(read_in_block), "+{s81}"(request_in_block),
                 "+{s[82:83]}"(entry_ptr), "+{s[84:85]}"(r.off1), "+{s[86:87]}"(r.off2), "+{s96}"(entry_requests),
                 "+{v208}"(entry)
               : TTPA_STREAM_COMMON_IN, "{s76}"(kv_heads), "{s77}"(kv_head), "{s78}"(num_blocks),
                 "{s79}"(tiles_per_block), "{s[98:99]}"(r.off0), "{s[50:51]}"(off1), "{s[52:53]}"(off2),
                 "{s54}"(entry0), "{s55}"(read_in_block0), "{s56}"(request_in_block0), "{s[58:59]}"(entry_ptr0)
               : "memory", "vcc", "scc", "m0", TTPA_STREAM_LOOP_CLOBBERS);
}

template <int HPW, int FORM>
__global__ __launch_bounds__(256, 2) void prefill_stream_kernel(PrefillArgs a) {
  constexpr int RPW = 4 / HPW;  // row blocks per workgroup
  constexpr int D = kD;
  constexpr bool PAGED = FORM == kPaged;
  using T = Tile<D>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  int wg = blockIdx.x;
  if constexpr (!PAGED) {
    wg = attention_workgroup<D>(a, wg);
    if (wg < 0) return;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int nqt = (a.sq + kRowsPerWave * RPW - 1) / (kRowsPerWave * RPW);
  const int groups = a.hq / HPW;
  const int xcd = wg & 7, slot = wg >> 3;
  const int yl = slot / a.spg;
  const int y = yl * 8 + xcd;
  if (y >= a.batch * groups) return;  // grid is padded to a multiple of 8 groups
  const int qt = nqt - 1 - (slot - yl * a.spg);
  const int b = y / groups;
  const int hq0 = (y - b * groups) * HPW;
  const int hk = hq0 / (a.hq / a.hkv);
  const int hq = hq0 + wave % HPW;
  const int row0 = (qt * RPW + wave / HPW) * kRowsPerWave;  // first query row of the wavefront
  const int offset = a.causal ? (a.chunk_start ? a.chunk_start[0] : 0) : 0;

  // keys the workgroup can see, in blocks of 32
  const int wg_last_row = min(a.sq, (qt + 1) * kRowsPerWave * RPW) - 1;
  const int kv_end = a.causal ? min(a.skv, offset + wg_last_row + 1) : a.skv;
  const int first_block = FORM == kDenseWindow ? max(0, offset + qt * kRowsPerWave * RPW - a.window + 1) / kBlockKeys : 0;
  const int nblk = __builtin_amdgcn_readfirstlane((kv_end + kBlockKeys - 1) / kBlockKeys - first_block);

  int spg = a.spg;
  if (a.spg_even > 0) {
    const int lightest = a.causal ? min(offset + kRowsPerWave, a.skv) : a.skv;
    const int heaviest = a.causal ? min(offset + a.sq, a.skv) : a.skv;
    if (4 * lightest >= 3 * heaviest) {
      spg = a.spg_even;
      if (slot - yl * a.spg >= spg) return;
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
    ldv[j] = (uint32_t)r * row_bytes + 16u * (uint32_t)(cp ^ T::swz_v(r)) + 1024u - 1024u * j;
  }
  sreq.m0_base = uni(lds0 + 2048u * (uint32_t)wave);
  sreq.k_requests = sreq.v_requests = nblk;
  sreq.off0 = sreq.off1 = sreq.off2 = 0;
  int entry = 0;
  uint64_t kbase0 = 0, vbase0 = 0;
  if constexpr (!PAGED) {
    const int64_t head = b * a.kv_bs + hk * a.kv_hs + (int64_t)first_block * kBlockKeys * a.kv_ts;
    kbase0 = uni(reinterpret_cast<uint64_t>(a.k + head) - 1024u);
    vbase0 = uni(reinterpret_cast<uint64_t>(a.v + head) - 1024u);
    sreq.kbase = kbase0, sreq.vbase = vbase0;
    sreq.stride = (uint32_t)(2 * kBlockKeys * a.kv_ts);
    stream_first_dense(sreq, ldk, ldv);
  } else {
    const int tpb = a.bs / kKeysPerTile, last = a.w * tpb - 1;  // (entries exist for every tile of the table)
    sreq.kbase = reinterpret_cast<uint64_t>(a.k) - 1024u;
    sreq.vbase = reinterpret_cast<uint64_t>(a.v) - 1024u;
    sreq.stride = (uint32_t)a.bs * (uint32_t)T::RB;
    int raw[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) raw[t] = a.pt[(int64_t)b * a.pt_rs + min(t, last) / tpb];
    uint64_t off[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      int phys = __builtin_amdgcn_readfirstlane(raw[t]);
      if ((unsigned)phys >= (unsigned)a.nb) phys = 0;
      off[t] = (uint64_t)((int64_t)phys * a.hkv + hk) * sreq.stride + (uint64_t)(min(t, last) % tpb) * T::TILE_BYTES;
    }
    sreq.off0 = uni(off[0]), sreq.off1 = uni(off[1]), sreq.off2 = uni(off[2]);
    entry = raw[3];
    stream_first_paged(sreq, ldk, ldv);
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
      vo[db] = lds0 + TTPA_STREAM_V_RING + (uint32_t)(vr * T::RB + 16 * (c ^ T::swz_v(vr)) + 8 * (a16 & 1));
    }
  }
  StreamItems it;
  it.k = 0, it.j = uni(slot - yl * a.spg), it.spg = uni(spg), it.nqt = uni(nqt);
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
  } else {
    const int tpb = a.bs / kKeysPerTile;
    stream_items_paged(sreq, it, q_lo, q_hi, ko, vo, ldk, ldv, q_base, out_base, n, 4 * h, a.scale_log2e, nblk, uni(a.hkv), uni(hk), uni(a.nb), uni(tpb), entry,
                       uni(reinterpret_cast<uint64_t>(a.pt + (int64_t)b * a.pt_rs + 4 / tpb)));
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
  if (HPW == 4 && FORM != kDenseWindow) {
    // Row blocks of nearly one weight (a chunk far into its sequence, or no causal mask) that fill the
    // chip more than once: one round of workgroups with equal shares instead, which saves the later
    // rounds' start-up (267 -> 261 us on 4 x 512-token chunks behind 4096 tokens, 64 heads).  The
    // chunk's start is in device memory, so the kernel decides: the workgroups past the round exit.
    int cus = device_cus();
    if (cus <= 0) cus = 256;
    const int one_round = (2 * cus + ny8 * 8 - 1) / (ny8 * 8);
    b.spg_even = one_round < nqt && nqt % one_round == 0 ? one_round : 0;
    if (const char *e = getenv("TTPA_PREFILL_WGS_PER_GROUP")) {  // (read on every call) an experiment's override
      if (atoi(e) > 0) b.spg = std::min(nqt, atoi(e)), b.spg_even = 0;
    }
  }
  int grid = b.spg * ny8 * 8;
  if (FORM != kPaged && a.fill_kc) grid = grid_with_fill(b, grid, kD);
  launch_dominant(&prefill_stream_kernel<HPW, FORM>, dim3(grid), dim3(256), (size_t)TTPA_STREAM_LDS_BYTES, st, b);
  return check_launch("sdpa_prefill");
}

template <int HPW>
int launch_heads(const PrefillArgs &a, hipStream_t st) {
  if (a.pt) return launch_form<HPW, kPaged>(a, st);
  return a.window > 0 ? launch_form<HPW, kDenseWindow>(a, st) : launch_form<HPW, kDense>(a, st);
}

}  // namespace

// The line lies where the loop's unit does: whole blocks of 32 keys that lie in one piece, at the one head
// size whose register map is built.  A dense K / V that ends inside a block, smaller cache blocks,
// windows over a paged cache and explicit masks are the plain loop's.  Wherever both run, this one is
// faster (above) or, on passes of a few microseconds, equal.
bool stream_serves(const PrefillArgs &a, int head_size) {
  if (!a.stream || head_size != kD || a.mask != nullptr) return false;
  if (a.pt) return a.bs % kKeysPerTile == 0 && a.window == 0;
  return a.skv % kBlockKeys == 0;
}

int launch_stream(const PrefillArgs &a, hipStream_t st) {
  const int g = a.hq / a.hkv;
  if (g % 4 == 0) return launch_heads<4>(a, st);
  if (g % 2 == 0) return launch_heads<2>(a, st);
  return launch_heads<1>(a, st);
}

}  // namespace ttpa
