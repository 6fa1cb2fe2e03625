// The streaming prefill kernel of one head size: included by prefill_stream.hip (128, and the choice) and
// prefill_stream_d64.hip / _d256.hip (a translation unit each: the blocks of assembly are long).
#pragma once

#include "prefill_parts.h"
#include "build/prefill_stream_asm.h"

#include <algorithm>
#include <cstdlib>

namespace ttpa {
namespace {

// kPaged: cache blocks of whole 64-key tiles (two 32-key blocks share a table entry); kPaged32: of whole
// 32-key blocks (an entry per block costs scalar instructions in every iteration, not in every other one)
// kDenseWide: keys of 128 + 64 features (the latent layers' prompts with K and V expanded per head): 20 matrix
// instructions per block of 32 keys; 4 x 2048 tokens, 16 heads: 8.6e10 flop in 100 us, where the absorbed form's
// 2.9e11 took 281
enum StreamForm { kDense = 0, kDenseWindow = 1, kPaged = 2, kPaged32 = 3, kDenseWide = 4 };

// The assembly is bound to the registers its text names through constraint strings (both written by
// gen_prefill_stream.py, with the names that the kernel below gives the values); everything else it
// touches is on the clobber list.  The requests of a workgroup's first blocks are a block of assembly of their own, issued right
// behind those of its Q rows so that the two round trips to memory overlap.  (Scalars only: with the per-lane
// offsets in the same struct the compiler keeps the whole of it in vector registers.)
struct StreamRequests {
  uint64_t kbase, vbase;       // dense: the first block of K / V; paged: the caches (both minus 1024 bytes)
  uint32_t stride;             // dense: bytes from a 32-key block to the next; paged: bytes of a (cache block, head) slab
  uint32_t m0_base;            // LDS address of the wavefront's first segment in K slot 0
  int k_requests, v_requests;  // blocks not requested yet
};

// Values the compiler may hold in vector registers although they are the same in every lane: the
// block binds them to scalar registers.
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint32_t uni(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
__device__ __forceinline__ uint64_t uni(uint64_t x) {
  return address_from_words(__builtin_amdgcn_readfirstlane((int)(uint32_t)x), __builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32)));
}

// The second part of the keys: its first block, bytes from a block to the next, the LDS address of the
// wavefront's segment, V's bytes per block, the lane's offset inside a block.
struct StreamWide {
  uint64_t base;
  uint32_t stride, m0, v_stride;
};

// What a workgroup works on (see gen_prefill_stream.py): which row blocks, and what the block of
// assembly needs to set one up.
struct StreamItems {
  int k, j, spg, nqt;          // item counter (starts at 0), the workgroup's slot, slots, row blocks
  int sq, skv, offset, causal;
  uint32_t q_row_bytes, out_row_bytes;
  int row0;                    // first query row of item 0
  int key0;                    // first key of its first block
};

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

// N 32-bit registers in a row, as the blocks of assembly take them.
template <int N>
struct Words {
  typedef uint32_t type __attribute__((ext_vector_type(N)));
  __device__ static __forceinline__ type of(const uint32_t (&x)[N]) {
    type w;
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = x[i];
    return w;
  }
};
template <>
struct Words<1> {
  typedef uint32_t type;
  __device__ static __forceinline__ type of(const uint32_t (&x)[1]) { return x[0]; }
};

// Workgroups of a CU by the registers of the blocks of assembly (168, 256, and 256 with 128 accumulation registers); LDS of one: rings of
// four or five blocks of K and of V, and for keys of 128 + 64 features of the second part.
constexpr int stream_wgs_per_cu(int d) { return d == 64 ? 3 : d == 128 ? 2 : 1; }
constexpr int stream_v_ring(int d, bool wide) { return TTPA_STREAM_SLOTS(d, wide) * kBlockKeys * 2 * d; }
constexpr int stream_p_ring(int d, bool wide) { return 2 * stream_v_ring(d, wide); }
constexpr int stream_lds_bytes(int d, bool wide) { return stream_p_ring(d, wide) + (wide ? TTPA_STREAM_SLOTS(d, wide) * kBlockKeys * 128 : 0); }

template <int D, int FORM>
__global__ __launch_bounds__(256, stream_wgs_per_cu(D)) void prefill_stream_kernel(PrefillArgs a) {
  constexpr bool PAGED = FORM == kPaged || FORM == kPaged32, WIDE = FORM == kDenseWide;
  using T = Tile<D>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  // The arguments that the set-up needs arrive as one batch (the compiler would wait for a first one to find the workgroup's place and then for
  // a second: a trip of a short pass's few), and the chunk's start is asked for before anything else is worked out.
  asm volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.pt), "s"(a.q_bs), "s"(a.q_hs), "s"(a.q_ts), "s"(a.pt_rs), "s"(a.out), "s"(a.out_bs),
               "s"(a.out_hs), "s"(a.out_ts), "s"(a.scale_log2e));
  if constexpr (!PAGED) asm volatile("" ::"s"(a.kv_bs), "s"(a.kv_hs), "s"(a.kv_ts));
  const int offset = a.causal ? chunk_offset(a.chunk_start, a.sq, a.skv) : 0;
  int wg = blockIdx.x;
  if constexpr (!PAGED && !WIDE) {
    wg = attention_workgroup<D>(a, wg);
    if (wg < 0) return;
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int nqt = (row_blocks(a) * a.head_group + 3) / 4;  // workgroups of a head group, one after the other in row blocks
  // The part is the slowest index: the workgroups of part 0, the only ones with work where the keys are few, are dealt over the
  // XCDs and CUs as in a launch that is not split.  (As the fastest index, they met on half of the CUs or a quarter: 256
  // workgroups over 512 keys 20.5 us, 16.3 this way.)
  const int part = PAGED ? blockIdx.y : 0;
  int y, item0;
  if (!workgroup_place(a, wg, y, item0)) return;
  const int qt = nqt - 1 - item0;
  const int b = quotient(a.by_groups, y);
  const int hq0 = (y - b * a.by_groups.d) * a.head_group;
  const int hk = quotient(a.by_group_heads, hq0);
  const int row_block = quotient(a.by_head_group, 4 * qt + wave);
  const int hq = hq0 + 4 * qt + wave - row_block * a.head_group;
  const int row0 = row_block * kRowsPerWave;  // first query row of the wavefront

  // keys the workgroup can see, in blocks of 32
  const int wg_last_row = min(a.sq, (last_row_block(a, qt) + 1) * kRowsPerWave) - 1;
  const int kv_end = a.causal ? min(a.skv, offset + wg_last_row + 1) : a.skv;
  int first_block = FORM == kDenseWindow ? max(0, offset + quotient(a.by_head_group, 4 * qt) * kRowsPerWave - a.window + 1) / kBlockKeys : 0;
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

  // ---- first requests: the Q rows, then the first blocks -------------------------------------------
  StreamRequests req;
  constexpr int LOADS = D / 64;  // of a wavefront per block and tensor
  uint32_t lane_k[LOADS], lane_v[LOADS];
  const uint32_t lds0 = lds_address(smem);
  const uint32_t row_bytes = PAGED ? (uint32_t)T::RB : 2u * (uint32_t)a.kv_ts;
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    // a block is 4 LOADS segments of 1 KiB; wavefront w requests segments LOADS w ...
    const int r = (LOADS * wave + j) * T::RPI + lane / T::CPR, cp = lane % T::CPR;
    lane_k[j] = (uint32_t)r * row_bytes + 16u * (uint32_t)(cp ^ T::swz_k(r)) + 1024u - 1024u * j;
    lane_v[j] = (uint32_t)r * (WIDE ? 2u * (uint32_t)a.v_ts : row_bytes) + 16u * (uint32_t)(cp ^ T::swz_v(r)) + 1024u - 1024u * j;
  }
  const auto ldk = Words<LOADS>::of(lane_k), ldv = Words<LOADS>::of(lane_v);
  // The wavefront's 32 Q rows, whole rows per load, go to the slot that K block ns - 1 (wavefront 0) or V block ns - 4 + wave takes later,
  // in the layout of a K block.  Loaded to registers by the lanes that hold them, 32 bytes of each of 32 rows per instruction, they cost a short pass
  // 0.65 us more.  (Where three of four wavefronts have no rows, one head per KV head and prompts of 32, the second trip through LDS, of the output,
  // cost as much again from five users on: 5 x 32 tokens of 16 / 16 heads of 128 5.72 / 5.80 us, 3 x 32 5.15 / 4.85.)
  constexpr int SLOTS = TTPA_STREAM_SLOTS(D, WIDE);
  const int q_slot = (wave == 0 ? SLOTS - 1 : 2 * SLOTS - 4 + wave) * (kBlockKeys * T::RB);
  {
    const uint16_t *qp = a.q + b * a.q_bs + hq * a.q_hs;
#pragma unroll
    for (int j = 0; j < kRowsPerWave / T::RPI; ++j) {
      const int r = j * T::RPI + lane / T::CPR;
      dma16_lane(qp + (int64_t)min(row0 + r, a.sq - 1) * a.q_ts + 8 * ((lane % T::CPR) ^ T::swz_k(r)), uni(lds0 + q_slot + 1024u * j));
    }
  }
  StreamWide wide;
  uint32_t ldp = 0;
  if constexpr (WIDE) {
    // a block of the second part is 4 segments of eight 128-byte rows, one per wavefront
    const int r = 8 * wave + (lane >> 3);
    ldp = (uint32_t)r * 2u * (uint32_t)a.k2_ts + 16u * (uint32_t)((lane & 7) ^ Tile<64>::swz_k(r));
    wide.base = uni(reinterpret_cast<uint64_t>(a.k2 + b * a.k2_bs + hk * a.k2_hs));
    wide.stride = (uint32_t)(2 * kBlockKeys * a.k2_ts), wide.v_stride = (uint32_t)(2 * kBlockKeys * a.v_ts);
    wide.m0 = uni(lds0 + stream_p_ring(D, WIDE) + 1024u * (uint32_t)wave);
  }
  req.m0_base = uni(lds0 + 1024u * LOADS * (uint32_t)wave);
  req.k_requests = req.v_requests = nblk;
  StreamTable tab;
  StreamPart out_part = {0, 0};
  uint64_t off[TTPA_STREAM_SLOTS(D, WIDE)];
  uint64_t kbase0 = 0, vbase0 = 0;
  if constexpr (!PAGED) {
    const int64_t head = b * a.kv_bs + hk * a.kv_hs + (int64_t)first_block * kBlockKeys * a.kv_ts;
    kbase0 = uni(reinterpret_cast<uint64_t>(a.k + head) - 1024u);
    vbase0 = uni(reinterpret_cast<uint64_t>(a.v + (WIDE ? b * a.v_bs + hk * a.v_hs : head)) - 1024u);
    req.kbase = kbase0, req.vbase = vbase0;
    req.stride = (uint32_t)(2 * kBlockKeys * a.kv_ts);
    if constexpr (WIDE) asm volatile(TTPA_STREAM_FIRST_DENSE_WIDE_128);
    else if constexpr (D == 64) asm volatile(TTPA_STREAM_FIRST_DENSE_64);
    else if constexpr (D == 128) asm volatile(TTPA_STREAM_FIRST_DENSE_128);
    else asm volatile(TTPA_STREAM_FIRST_DENSE_256);
  } else {
    // keys that share a table entry are a multiple of a unit (a 64-key tile, a 32-key block); the first FIRST
    // units are requested here, the loop takes raw entries from there on
    constexpr int UNIT = FORM == kPaged ? kKeysPerTile : kBlockKeys;
    constexpr int FIRST = FORM == kPaged ? (SLOTS + 1) / 2 : SLOTS, RAW = FORM == kPaged ? 1 : 2;
    const int per = a.bs / UNIT, last = a.w * per - 1;  // (entries exist for every unit of the table)
    const int unit0 = first_block * kBlockKeys / UNIT;
    auto column = [&](int unit) { return div_block(a, unit * UNIT); };
    auto in_block = [&](int unit) { return unit - column(unit) * per; };
    req.kbase = reinterpret_cast<uint64_t>(a.k) - 1024u;
    req.vbase = reinterpret_cast<uint64_t>(a.v) - 1024u;
    req.stride = (uint32_t)a.bs * (uint32_t)T::RB;
    int raw[FIRST + RAW];
#pragma unroll
    for (int t = 0; t < FIRST + RAW; ++t) raw[t] = a.pt[(int64_t)b * a.pt_rs + column(min(unit0 + t, last))];
#pragma unroll
    for (int t = 0; t < FIRST; ++t) {
      int phys = __builtin_amdgcn_readfirstlane(raw[t]);
      if ((unsigned)phys >= (unsigned)a.nb) phys = 0;
      off[t] = uni((uint64_t)((int64_t)phys * a.hkv + hk) * req.stride + (uint64_t)in_block(min(unit0 + t, last)) * (UNIT * T::RB));
    }
    tab.kv_heads = uni(a.hkv), tab.kv_head = uni(hk), tab.num_blocks = uni(a.nb), tab.per_block = uni(per);
    tab.entry = raw[FIRST], tab.entry2 = raw[FIRST + RAW - 1];
    const int next = unit0 + FIRST;
    tab.read_in_block = uni(in_block(next)), tab.request_in_block = uni(in_block(next + RAW));
    tab.entry_ptr = uni(reinterpret_cast<uint64_t>(a.pt + (int64_t)b * a.pt_rs + column(next + RAW)));
    tab.entry_requests = uni(max((nblk - 1) / (UNIT / kBlockKeys) + 1 - FIRST - RAW, 0));
    if constexpr (FORM == kPaged && D == 64) asm volatile(TTPA_STREAM_FIRST_PAGED_64);
    else if constexpr (FORM == kPaged && D == 128) asm volatile(TTPA_STREAM_FIRST_PAGED_128);
    else if constexpr (FORM == kPaged) asm volatile(TTPA_STREAM_FIRST_PAGED_256);
    else if constexpr (D == 64) asm volatile(TTPA_STREAM_FIRST_PAGED32_64);
    else if constexpr (D == 128) asm volatile(TTPA_STREAM_FIRST_PAGED32_128);
    else asm volatile(TTPA_STREAM_FIRST_PAGED32_256);
    if (!whole && row0 < a.sq) {
      const PartLayout lay = part_layout(a);
      const int64_t at = (((int64_t)part * a.batch + b) * a.hq + hq) * lay.row_blocks + row_block;
      out_part.acc = uni(reinterpret_cast<uint64_t>(a.part_acc + at * part_acc_floats(D)));
      out_part.stats = uni(reinterpret_cast<uint64_t>(a.part_acc + lay.slots * part_acc_floats(D) + at * (2 * kRowsPerWave)));
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
      po[s] = lds0 + stream_p_ring(D, WIDE) + (uint32_t)(n * 128 + 16 * ((2 * s + h) ^ Tile<64>::swz_k(n)));
    }
  }
  // LDS operand addresses of the lane inside slot 0 of the K ring and of the V ring: K fragment of k-step
  // s, V^T fragment of output block db (through the transposing LDS load; the layout of prefill.hip)
  uint32_t lane_ko[D / 16], lane_vo[D / 32];
#pragma unroll
  for (int s = 0; s < D / 16; ++s) lane_ko[s] = lds0 + (uint32_t)(n * T::RB + 16 * ((2 * s + h) ^ T::swz_k(n)));
  {
    const int grp = lane >> 4, a16 = lane & 15, vr = 4 * (grp >> 1) + (a16 >> 2);
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      const int c = 4 * db + 2 * (grp & 1) + ((a16 & 3) >> 1);
      lane_vo[db] = lds0 + stream_v_ring(D, WIDE) + (uint32_t)(vr * T::RB + 16 * (c ^ T::swz_v(vr)) + 8 * (a16 & 1));
    }
  }
  const auto ko = Words<D / 16>::of(lane_ko);
  const auto vo = Words<D / 32>::of(lane_vo);
  StreamItems it;
  it.k = 0, it.j = uni(item0), it.spg = uni(spg), it.nqt = uni(nqt);
  it.sq = uni(a.sq), it.skv = uni(a.skv), it.offset = uni(offset), it.causal = uni(a.causal);
  it.q_row_bytes = uni(2u * (uint32_t)a.q_ts), it.out_row_bytes = uni(2u * (uint32_t)a.out_ts);
  it.row0 = __builtin_amdgcn_readfirstlane(row0);
  it.key0 = uni(first_block * kBlockKeys);
  const int out_slot = wave * (kBlockKeys * T::RB);
  const uint32_t out_address = uni(lds0 + out_slot);
  const uint64_t out_row0 = uni(reinterpret_cast<uint64_t>(a.out + b * a.out_bs + hq * a.out_hs));
  // per lane: row 0 of the lane's head, at the lane's 8 (lane / 32) elements
  const uint64_t q_base = reinterpret_cast<uint64_t>(a.q + b * a.q_bs + hq * a.q_hs + 8 * h);
  const uint64_t out_base = reinterpret_cast<uint64_t>(a.out + b * a.out_bs + hq * a.out_hs + 8 * h);
  const int h4 = 4 * h;
  int lowest = 0, low_to = 0;
  if constexpr (FORM == kDenseWindow) {
    lowest = offset + min(row0 + n, a.sq - 1) - a.window + 1 - h4;
    low_to = uni(offset + row0 + kRowsPerWave - a.window);
  }
  // Everything behind the first requests of item 0, through the stored output rows of the last item.
  if constexpr (WIDE) asm volatile(TTPA_STREAM_LOOP_DENSE_WIDE_128);
  else if constexpr (FORM == kDense && D == 64) asm volatile(TTPA_STREAM_LOOP_DENSE_64);
  else if constexpr (FORM == kDense && D == 128) asm volatile(TTPA_STREAM_LOOP_DENSE_128);
  else if constexpr (FORM == kDense) asm volatile(TTPA_STREAM_LOOP_DENSE_256);
  else if constexpr (FORM == kDenseWindow && D == 64) asm volatile(TTPA_STREAM_LOOP_DENSE_WINDOW_64);
  else if constexpr (FORM == kDenseWindow && D == 128) asm volatile(TTPA_STREAM_LOOP_DENSE_WINDOW_128);
  else if constexpr (FORM == kDenseWindow) asm volatile(TTPA_STREAM_LOOP_DENSE_WINDOW_256);
  else if constexpr (FORM == kPaged && D == 64) asm volatile(TTPA_STREAM_LOOP_PAGED_64);
  else if constexpr (FORM == kPaged && D == 128) asm volatile(TTPA_STREAM_LOOP_PAGED_128);
  else if constexpr (FORM == kPaged) asm volatile(TTPA_STREAM_LOOP_PAGED_256);
  else if constexpr (D == 64) asm volatile(TTPA_STREAM_LOOP_PAGED32_64);
  else if constexpr (D == 128) asm volatile(TTPA_STREAM_LOOP_PAGED32_128);
  else asm volatile(TTPA_STREAM_LOOP_PAGED32_256);
}

template <int D, int FORM>
int launch_form(const PrefillArgs &a, hipStream_t st) {
  constexpr int lds = stream_lds_bytes(D, FORM == kDenseWide);
  constexpr bool PAGED = FORM == kPaged || FORM == kPaged32;
  static std::atomic<uint64_t> lds_ready{0};
  if (!ensure_dynamic_lds(reinterpret_cast<const void *>(&prefill_stream_kernel<D, FORM>), lds, lds_ready))
    return fail(TTPA_ERR_LAUNCH, "prefill: cannot reserve %d bytes of LDS", lds);
  PrefillArgs b = a;
  b.spg_even = 0, b.parts = 1;
  const int heads = head_group_size(a, D);
  // One workgroup per row block and head group, heavy blocks first, and the dispatcher deals them to the CUs
  // as slots free up: the loop can also give a workgroup several row blocks (spg workgroups per group,
  // TTPA_PREFILL_WGS_PER_GROUP), but one round of two workgroups per CU measured 204 us against 150 on
  // the 4 x 2048-token causal workload (a change of row block costs a workgroup about 4 us in which
  // nothing of its own overlaps, and a static deal cannot make up for workgroups that start late).
  const bool items = D == 128 && heads == 4 && (FORM == kDense || FORM == kPaged);  // the loop can go on with another row block
  // (read on every call) an experiment's override: several row blocks per workgroup, each over all of its keys
  const char *e = items ? getenv("TTPA_PREFILL_WGS_PER_GROUP") : nullptr;
  const int per_group = e ? atoi(e) : 0;
  if (PAGED && per_group <= 0 && a.part_acc && a.part_bytes >= part_bytes(a, heads, stream_split(D), D)) set_parts(b, heads, stream_split(D));
  int grid = lay_out(b, heads, 0, PAGED && spreads_groups(b, heads, D));
  if (per_group > 0) {
    grid = lay_out(b, heads, std::min(b.spg, per_group));
  } else if (items && b.parts == 1) {
    // Row blocks of nearly one weight (a chunk far into its sequence, or no causal mask) that fill the
    // chip more than once: one round of workgroups with equal shares instead, which saves the later
    // rounds' start-up (267 -> 261 us on 4 x 512-token chunks behind 4096 tokens, 64 heads).  The
    // chunk's start is in device memory, so the kernel decides: the workgroups past the round exit.
    const int groups = a.batch * (a.hq / heads), one_round = (2 * a.cus + groups - 1) / groups;
    b.spg_even = one_round < b.spg && b.spg % one_round == 0 ? one_round : 0;
  }
  if (!PAGED && FORM != kDenseWide && a.fill_kc) grid = grid_with_fill(b, grid, D);
  launch_dominant(&prefill_stream_kernel<D, FORM>, dim3(grid, b.parts), dim3(256), (size_t)lds, st, b);
  if (const int rc = check_launch("sdpa_prefill")) return rc;
  if (b.parts > 1) {
    prefill_merge_kernel<D><<<dim3((b.sq + kRowsPerWave - 1) / kRowsPerWave, b.hq, b.batch), dim3(2 * D), 0, st>>>(b);
    return check_launch("sdpa_prefill (merge of the parts)");
  }
  return TTPA_OK;
}

template <int D>
int launch_stream_d(const PrefillArgs &a, hipStream_t st) {
  if (a.pt) return a.bs % kKeysPerTile == 0 ? launch_form<D, kPaged>(a, st) : launch_form<D, kPaged32>(a, st);
  return a.window > 0 ? launch_form<D, kDenseWindow>(a, st) : launch_form<D, kDense>(a, st);
}

}  // namespace
}  // namespace ttpa
