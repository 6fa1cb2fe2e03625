// Prefill attention (dense and paged / chunked) on bf16 MFMA tiles, gfx950.
//
// One workgroup = 4 wavefronts that share every K/V tile in LDS.  A wavefront owns a
// block of 32 query rows of one query head; the 4 wavefronts are HPW heads of the same
// KV head times 4 / HPW consecutive row blocks, so with grouped heads a K/V tile is
// fetched once for up to 4 query heads.
//
// Per 64-key tile a wavefront computes, with v_mfma_f32_32x32x16_bf16:
//   S^T[key, row] = K[key, :] . Q[row, :]      A = K tile rows (LDS), B = Q (registers)
//   O^T[d, row]  += V^T[d, key] . P^T[key, row] A = V tile read through the transposing
//                                               LDS load, B = P^T (registers)
// Computing the TRANSPOSED score tile puts one query row in each lane's accumulator
// column: the online-softmax statistics of a row are plain per-lane scalars (one
// exchange between the two lane halves per tile), and the probabilities a lane holds are
// exactly the B-operand fragment the second product needs, so P never moves between
// lanes or through LDS.
//
// Accumulator layout of a 32x32 tile (lane = 32 h + n): register r holds
// element (row 8 (r / 4) + 4 h + r % 4, column n).
//
// K/V tiles travel global memory -> LDS directly (global_load_lds_dwordx4: 64 lanes x 16
// bytes land in 1 KiB of consecutive LDS), with no staging registers.  Rows are therefore
// unpadded in LDS; bank conflicts are avoided by an XOR swizzle of the 16-byte chunk
// position inside a row, applied on the global side (which chunk a lane fetches) and again
// when fragments are read.
#include "prefill_parts.h"

#include <algorithm>
#include <cstdlib>

namespace ttpa {
namespace {

// v_max3_f32 without the input canonicalisation the compiler adds around fmaxf (scores are
// never signalling NaNs).  Callers order it after a compiler-visible read of the matrix
// results, which is where the matrix-to-vector hazard wait states are inserted.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float d;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}

// Expansion of the block-float-8 blocks a chunk pass reads into bfloat16 copies, so that the
// hand-scheduled loop (which wants bfloat16 blocks it can request straight into LDS) serves a
// block-float-8 cache too: the slab of table entry x = batch entry * width + column and of a (KV head, K or V)
// goes to block x of a scratch cache, and entry x of the identity table that goes with it is written.  Memory work (1 byte
// in, 2 out per element) of about a tenth of the attention's time.  How many columns the pass reads is in device memory, so
// a fixed number of workgroups (eight per CU, what fits) walks the slabs there are: one workgroup per slab of the page table cost
// 0.25 ns each where most had nothing to do (4 x 64 rows behind 256 tokens, 16 / 16 heads, blocks of 32 under 32768 columns:
// the pass 60.9 -> 25.4 us).
constexpr int kExpandWorkgroups = 2048;
struct ExpandArgs {
  const uint8_t *kc, *vc;  // the block-float-8 caches
  uint16_t *k, *v;         // scratch caches [batch * width][KV heads][block size][D]
  int32_t *table;          // [batch][width]
  const int32_t *pt;
  int64_t pt_rs;
  const int32_t *chunk_start;
  int batch, w, hkv, bs, nb, sq, causal;
  Divisor by_pieces, by_slabs;  // pieces of a slab, slabs of a block
};

// Bound by memory.  A wavefront's piece is 64 groups in halves: 8 bytes of a half become 16, so that an instruction writes 1 KiB in
// one piece; it asks for its next piece before it writes the one it has.  3 x 992 rows behind 1024 tokens of 8 heads of 128 (37 MB) 12.0 -> 9.4 us,
// 3 x 1728 behind 4096 (110 MB) 27.3 -> 22.3, against a workgroup per slab in turn and 16 bytes of every 32 per store (10.2 and 26.3 with
// whole groups); the passes 71.3 -> 68.5 and 272.6 -> 271.3, for of the copies that exceed the caches the attention waits for what is left
// to write.
template <int D>
__global__ __launch_bounds__(256) void bfp8_expand_kernel(ExpandArgs e) {
  const int skv = e.w * e.bs;
  const int kv_end = e.causal ? min(skv, chunk_offset(e.chunk_start, e.sq, skv) + e.sq) : skv;
  const int cols = (kv_end + e.bs - 1) / e.bs;  // page-table columns that the pass reads
  const int pieces = kv_end > 0 ? e.batch * cols * e.by_slabs.d * e.by_pieces.d : 0;
  const int lane = threadIdx.x & 63;
  struct Piece {
    uint2 bytes[2];
    uint32_t exponent[2];
    uint16_t *dst;
  };
  auto request = [&](int at) {
    const int item = quotient(e.by_pieces, at), r = quotient(e.by_slabs, item);  // slab and block of the pass
    const int part = item - r * e.by_slabs.d, b = r / cols, j = r - b * cols, x = b * e.w + j;
    const bool is_v = part >= e.hkv;
    const int h = part - (is_v ? e.hkv : 0), half = 128 * (at - item * e.by_pieces.d) + lane;
    int phys = e.pt[(int64_t)b * e.pt_rs + j];
    if ((unsigned)phys >= (unsigned)e.nb) phys = 0;  // (as the attention kernels treat a bad entry)
    if (part == 0 && half == 0) e.table[x] = x;
    const uint8_t *src = (is_v ? e.vc : e.kc) + ((int64_t)phys * e.hkv + h) * ((int64_t)(e.bs + e.bs / 16) * D);
    Piece p;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      p.bytes[i] = *reinterpret_cast<const uint2 *>(src + 8 * (half + 64 * i));
      p.exponent[i] = src[(int64_t)e.bs * D + (half + 64 * i) / 2];
    }
    p.dst = (is_v ? e.v : e.k) + ((int64_t)x * e.hkv + h) * e.bs * D + 8 * half;
    return p;
  };
  const int step = (int)gridDim.x * 4;
  int at = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (at >= pieces) return;
  Piece p = request(at);
  for (;;) {
    at += step;
    const bool more = at < pieces;
    Piece next = p;
    if (more) next = request(at);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float sc = bfp8_group_scale(p.exponent[i]), off = -128.f * sc;
      u32x4 out;
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const uint32_t v = w ? p.bytes[i].y : p.bytes[i].x;
        const float f0 = fmaf((float)(v & 0xffu), sc, off), f1 = fmaf((float)((v >> 8) & 0xffu), sc, off);
        const float f2 = fmaf((float)((v >> 16) & 0xffu), sc, off), f3 = fmaf((float)(v >> 24), sc, off);
        // the products are exact in bfloat16: their upper halves are the elements
        out[2 * w] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f1), __builtin_bit_cast(uint32_t, f0), 0x07060302u);
        out[2 * w + 1] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f3), __builtin_bit_cast(uint32_t, f2), 0x07060302u);
      }
      *reinterpret_cast<u32x4 *>(p.dst + 512 * i) = out;
    }
    if (!more) return;
    p = next;
  }
}

// MODE 0: dense K/V; 1: paged, block_size a multiple of 64 (a tile lies in one block);
// 3: paged, block_size a multiple of the rows one wavefront load covers (1 KiB: 8 / 4 / 2 rows
// for head sizes 64 / 128 / 256): one wavefront-uniform table lookup per load; 2: paged, any
// block size (per-lane table lookups); 4: paged block-float-8 caches (block_size a multiple of
// 16).  In mode 4 a tile goes global -> registers -> LDS: a thread fetches groups of 16 element
// bytes with their exponent byte (D / 64 groups per tile and tensor) where the other modes issue
// their LDS-DMA loads, and expands them to bfloat16 (exact: a 7-bit magnitude times a power of
// two) into the same swizzled tile layout at the end of the iteration, one tile period before
// the tile is used.  One workgroup per CU: the staging registers do not fit next to a second one.
//
// Per-tile schedule of a workgroup (LDS holds two K stages and two V stages):
//   S^T = K(t) Q^T | barrier | issue loads of K(t+2) and V(t+1) | softmax | O^T += V(t)^T P^T
// Every load is issued right after a barrier and has to have landed by the next one, one
// whole tile later.  K(t+2) overwrites the stage of K(t), which everybody has finished
// reading at the barrier of tile t; V(t+1) overwrites the stage of V(t-1), read before that
// barrier too.  LDS operand reads run a few fragments ahead of the matrix instructions that
// consume them.
//
// A wavefront has one block of 32 query rows, as workgroup_place and the parts know it (two, one workgroup per CU and every K / V
// fragment feeding two matrix instructions, measured slower: with one wavefront per SIMD nobody fills the waits for fragments and barriers).
//
// SPLIT: the keys of a row block are shared by a.parts > 1 workgroups (prefill_parts.h).  A kernel of its own: with the parts' way
// out as a run-time branch an unsplit launch was 0.1 ... 0.7 us longer than without (1 x 512 rows of 64 / 8 heads of 64 behind 512
// tokens 28.3 / 27.7 us, 8 x 256 of 16 / 8 of 256 behind 512 55.3 / 54.3), and a split one 0.3 us (1 x 32 of 16 / 8 of 256 22.5 / 22.2).
constexpr int prefill_wgs_per_cu(int d) { return d <= 128 ? 2 : 1; }

template <int D, int HPW, int MODE, bool SPLIT>
__global__ __launch_bounds__(256, prefill_wgs_per_cu(D)) void prefill_kernel(PrefillArgs a) {
  constexpr int RPW = 4 / HPW;            // wavefront row slots per workgroup
  constexpr int RH = 1;                   // blocks of query rows per wavefront
  constexpr int ROWS = kRowsPerWave * RH;
  constexpr int KSTEPS = D / 16;          // MFMA k-steps over the head dimension
  constexpr int DBLK = D / 32;            // 32-wide output blocks over the head dimension
  using T = Tile<D>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  int wg = blockIdx.x;  // index among the attention workgroups
  if constexpr (MODE == 0) {
    wg = attention_workgroup<D>(a, wg);
    if (wg < 0) return;
  }
  // (the slower index, so that part 0, alone with work where the keys are few, is on every XCD)
  const int part = SPLIT ? blockIdx.y : 0;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int n_lane = n;
  const int nqt = (a.sq + ROWS * RPW - 1) / (ROWS * RPW);
  int y, rank;
  if (!workgroup_place(a, wg, y, rank)) return;
  const int qt = nqt - 1 - rank;  // heavy (late) tiles are scheduled first
  const int b = quotient(a.by_groups, y);
  const int hq0 = (y - b * a.by_groups.d) * HPW;
  const int hk = quotient(a.by_group_heads, hq0);
  const int hq = hq0 + wave % HPW;
  const int row0 = (qt * RPW + wave / HPW) * ROWS;  // first query row of the wavefront
  // (the dense form has no chunk_start and at least one tile: without the bounds its code is what it was, 2 % faster at head size 256)
  const int offset = !a.causal ? 0 : MODE != 0 ? chunk_offset(a.chunk_start, a.sq, a.skv) : a.chunk_start ? a.chunk_start[0] : 0;

  // keys this workgroup / this wavefront can see
  const int wg_last_row = min(a.sq, (qt + 1) * ROWS * RPW) - 1;
  const int kv_end_wg = a.causal ? min(a.skv, offset + wg_last_row + 1) : a.skv;
  // (at least one tile: where no row sees a key, tile 0 is read and no score of it is computed)
  int ntiles = (kv_end_wg + kKeysPerTile - 1) / kKeysPerTile;
  if (MODE != 0) ntiles = max(ntiles, 1);
  const int wave_last_key = a.causal ? offset + min(a.sq - 1, row0 + ROWS - 1) : a.skv - 1;
  const bool wave_active = row0 < a.sq;
  // sliding window: first key any row of the workgroup / of this wavefront can see
  const int wg_first_key = a.window > 0 ? max(0, offset + qt * ROWS * RPW - a.window + 1) : 0;
  const int wave_first_key = a.window > 0 ? max(0, offset + row0 - a.window + 1) : 0;
  int first_tile = wg_first_key / kKeysPerTile;
  bool whole = true;  // this workgroup sees all keys of its rows
  if constexpr (SPLIT) {  // (no window, no mask)
    const int share = __builtin_amdgcn_readfirstlane((blocks_per_part(a, offset) + 1) / 2);
    whole = share >= ntiles;
    first_tile = part * share;
    ntiles = min(ntiles, first_tile + share);
    if (first_tile >= ntiles) return;
  }

  // ---- Q fragments (B operand: lane n = query row, 8 head-dim elements per k-step) -----
  bf16x8 qf[RH][KSTEPS];
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) {
    const int qrow = min(row0 + n, a.sq - 1);
    const uint16_t *qp = a.q + b * a.q_bs + hq * a.q_hs + (int64_t)qrow * a.q_ts + 8 * h;
    qf[0][s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(qp + 16 * s));
  }

  floatx16 acc[RH][DBLK];
  float m_run[RH], l_run[RH];
#pragma unroll
  for (int x = 0; x < RH; ++x) {
    m_run[x] = -INFINITY, l_run[x] = 0.f;
#pragma unroll
    for (int i = 0; i < DBLK; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][i][r] = 0.f;
  }

  // ---- global -> LDS tile loads ----------------------------------------------------------
  // Load j of this wavefront fills LDS segment 4 j + wave of a tile: RPI whole rows.  Lane l
  // writes chunk position l % CPR of row seg * RPI + l / CPR, so it fetches logical chunk
  // (l % CPR) ^ swz(row).  The per-lane part of the source address is fixed for all tiles.
  int ld_row[T::NI];       // row inside the tile
  uint32_t ld_k[T::NI], ld_v[T::NI];  // byte offset of the lane's chunk inside a tile (modes 0 and 1)
#pragma unroll
  for (int j = 0; j < T::NI; ++j) {
    const int r = (4 * j + wave) * T::RPI + lane / T::CPR;
    const int cp = lane % T::CPR;
    const uint32_t row_bytes = MODE == 0 ? 2u * (uint32_t)a.kv_ts : (uint32_t)T::RB;
    ld_row[j] = r;
    ld_k[j] = (uint32_t)r * row_bytes + 16u * (uint32_t)(cp ^ T::swz_k(r));
    ld_v[j] = (uint32_t)r * row_bytes + 16u * (uint32_t)(cp ^ T::swz_v(r));
  }
  // Issues the loads of one tile of one tensor.  Keys past the end of K/V are clamped to the
  // last row, whose scores are masked and whose V rows therefore carry weight 0.
  // Modes 1 and 3 look their blocks up one tile ahead of the loads (below): NLK wavefront-
  // uniform table entries per tile, one for the whole tile or one per load of this wavefront.
  constexpr int GPR = D / 16;           // mode 4: 16-element groups (= exponent bytes) per row
  constexpr int NG = D / 64;            // mode 4: groups per thread, tile and tensor
  constexpr int NLK = MODE == 1 ? 1 : (MODE == 3 ? T::NI : (MODE == 4 ? NG : 0));
  struct Blocks {
    int phys[NLK > 0 ? NLK : 1];
  };
  // first key of lookup j of tile kt
  auto lookup_key = [&](int kt, int j) {
    const int key0 = kt * kKeysPerTile;
    if constexpr (MODE == 1) return key0;
    if constexpr (MODE == 4) return key0 + min((tid + 256 * j) / GPR, a.skv - 1 - key0);  // per lane
    // the rows of a load sit in one block; a load wholly past the last key reads the rows that
    // hold the last key again (readable, and masked like any key past the end)
    return key0 + min((4 * j + wave) * T::RPI, (a.skv - 1 - key0) / T::RPI * T::RPI);
  };
  // LDS byte offset of a tile: stages of a K and a V tile each
  auto tile_offset = [&](bool is_v, int buf) { return (uint32_t)(buf * T::STAGE_BYTES + (is_v ? T::TILE_BYTES : 0)); };
  auto issue = [&](const uint16_t *src, const uint32_t (&ld)[T::NI], bool is_v, int kt, int buf,
                   const Blocks &blk) {
    const int key0 = kt * kKeysPerTile;
    const int last = a.skv - 1 - key0;  // last valid key of this tile, relative (>= 0)
    const uint32_t lds_base = lds_address(smem) + tile_offset(is_v, buf);
    const char *base = nullptr;  // uniform address of the tile (modes 0 and 1)
    if constexpr (MODE == 0) {
      base = reinterpret_cast<const char *>(src + b * a.kv_bs + hk * a.kv_hs + (int64_t)key0 * a.kv_ts);
    } else if constexpr (MODE == 1) {
      base = reinterpret_cast<const char *>(
          src + (((int64_t)blk.phys[0] * a.hkv + hk) * a.bs + (key0 - div_block(a, key0) * a.bs)) * D);
    }
    auto lds_dst = [&](int j) { return lds_base + (uint32_t)(4 * j + wave) * 1024u; };
    if constexpr (MODE == 2) {
#pragma unroll
      for (int j = 0; j < T::NI; ++j) {
        const int key = key0 + min(ld_row[j], last);
        const int col = div_block(a, key);
        int phys = a.pt[(int64_t)b * a.pt_rs + col];
        if ((unsigned)phys >= (unsigned)a.nb) phys = 0;
        const int c = (lane % T::CPR) ^ (is_v ? T::swz_v(ld_row[j]) : T::swz_k(ld_row[j]));
        dma16_lane(src + (((int64_t)phys * a.hkv + hk) * a.bs + (key - col * a.bs)) * D + c * 8, lds_dst(j));
      }
    } else if constexpr (MODE == 3) {
#pragma unroll
      for (int j = 0; j < T::NI; ++j) {
        const int key = lookup_key(kt, j);
        const char *seg = reinterpret_cast<const char *>(
            src + (((int64_t)blk.phys[j] * a.hkv + hk) * a.bs + (key - div_block(a, key) * a.bs)) * D);
        dma16(seg, ld[j] - (uint32_t)((4 * j + wave) * T::RPI * T::RB), lds_dst(j));
      }
    } else if (MODE == 0 && last < kKeysPerTile - 1) {  // uniform: dense K/V ending inside the tile
#pragma unroll
      for (int j = 0; j < T::NI; ++j) {
        const int c = (lane % T::CPR) ^ (is_v ? T::swz_v(ld_row[j]) : T::swz_k(ld_row[j]));
        const uint32_t off = (uint32_t)min(ld_row[j], last) * 2u * (uint32_t)a.kv_ts + 16u * (uint32_t)c;
        dma16(base, off, lds_dst(j));
      }
    } else {
#pragma unroll
      for (int j = 0; j < T::NI; ++j) dma16(base, ld[j], lds_dst(j));
    }
  };
  // ---- mode 4: block-float-8 tiles through registers --------------------------------------
  struct Staged {
    u32x4 bytes[MODE == 4 ? NG : 1];
    uint32_t ex[MODE == 4 ? NG : 1];
  };
  // group j of this thread: row (tid + 256 j) / GPR of the tile, 16 elements from 16 ((tid + 256 j) % GPR)
  auto fetch_bfp8 = [&](const uint16_t *cache, int kt, const Blocks &blk) {
    Staged st = {};
    if constexpr (MODE == 4) {
      const uint8_t *base = reinterpret_cast<const uint8_t *>(cache);
      const int64_t slab = (int64_t)(a.bs + a.bs / 16) * D;
#pragma unroll
      for (int j = 0; j < NG; ++j) {
        const int key = lookup_key(kt, j), c16 = (tid + 256 * j) % GPR;
        const int rowin = key - div_block(a, key) * a.bs;
        const uint8_t *sl = base + ((int64_t)blk.phys[j] * a.hkv + hk) * slab;
        st.bytes[j] = *reinterpret_cast<const u32x4 *>(sl + rowin * D + 16 * c16);
        st.ex[j] = sl[(int64_t)a.bs * D + rowin * GPR + c16];
      }
    }
    return st;
  };
  // (b - 128) * 2^(e - 133) for the 16 bytes of a group, as 8 bfloat16 pairs; LDS chunks
  // 2 c16 and 2 c16 + 1 of the row, at their swizzled positions
  auto commit_bfp8 = [&](const Staged &st, bool is_v, int buf) {
    if constexpr (MODE == 4) {
      unsigned char *tile_base = smem + buf * T::STAGE_BYTES + (is_v ? T::TILE_BYTES : 0);
#pragma unroll
      for (int j = 0; j < NG; ++j) {
        const int row = (tid + 256 * j) / GPR, c16 = (tid + 256 * j) % GPR;
        const float sc = bfp8_group_scale(st.ex[j]), off = -128.f * sc;
        uint32_t o[8];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint32_t x = st.bytes[j][w];
          const float f0 = fmaf((float)(x & 0xffu), sc, off), f1 = fmaf((float)((x >> 8) & 0xffu), sc, off);
          const float f2 = fmaf((float)((x >> 16) & 0xffu), sc, off), f3 = fmaf((float)(x >> 24), sc, off);
          // the products are exact in bfloat16: their upper halves are the elements
          o[2 * w] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f1), __builtin_bit_cast(uint32_t, f0), 0x07060302u);
          o[2 * w + 1] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f3), __builtin_bit_cast(uint32_t, f2), 0x07060302u);
        }
        const int sw = is_v ? T::swz_v(row) : T::swz_k(row);
        unsigned char *rp = tile_base + row * T::RB;
        *reinterpret_cast<uint4 *>(rp + 16 * ((2 * c16) ^ sw)) = make_uint4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<uint4 *>(rp + 16 * ((2 * c16 + 1) ^ sw)) = make_uint4(o[4], o[5], o[6], o[7]);
      }
    }
  };
  auto wait_loads_and_sync = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's tile loads have landed
    __syncthreads();
  };

  // ---- LDS operand addresses of this lane inside a stage (bytes) ------------------------
  uint32_t koff[KSTEPS];  // K fragment of k-step s, key block 0 (key block 1: + 32 rows)
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s)
    koff[s] = (uint32_t)(n * T::RB + 16 * ((2 * s + h) ^ T::swz_k(n)));
  // V^T fragment: through the transposing LDS load, per group of 16 lanes, lane i receives
  // element i % 4 of the 8-byte chunks addressed by lanes 4 j + i / 4.  This lane addresses
  // row 4 (grp / 2) + a16 / 4 (+ 16 per key step, + 8 for the second half), elements
  // 32 db + 16 (grp % 2) + 4 (a16 % 4).
  const int grp = lane >> 4, a16 = lane & 15;
  uint32_t voff[DBLK];
  {
    const int vr = 4 * (grp >> 1) + (a16 >> 2);
#pragma unroll
    for (int db = 0; db < DBLK; ++db) {
      const int c = 4 * db + 2 * (grp & 1) + ((a16 & 3) >> 1);
      voff[db] = (uint32_t)(vr * T::RB + 16 * (c ^ T::swz_v(vr)) + 8 * (a16 & 1));
    }
  }
  // K fragment i of a tile in issue order: k-step i / 2 of key block i % 2 (the two score
  // blocks alternate so consecutive matrix instructions are independent).
  auto read_k = [&](const unsigned char *st_base, int i) -> bf16x8 {
    const int s = i >> 1, kb = i & 1;
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(st_base + koff[s] + 32 * kb * T::RB));
  };
  // V^T fragment j in issue order: key step j / DBLK, output block j % DBLK (st_base: the V tile).
  auto read_v = [&](const unsigned char *st_base, int j) -> bf16x8 {
    typedef __attribute__((address_space(3))) shortx4 *lds_v4;
    const int k4 = j / DBLK, db = j % DBLK;
    const unsigned char *vk = st_base + voff[db] + 16 * k4 * T::RB;
    shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(vk));
    shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(vk + 8 * T::RB));
    bf16x4 l4 = __builtin_bit_cast(bf16x4, lo), h4 = __builtin_bit_cast(bf16x4, hi);
    bf16x8 t;
    t[0] = l4[0], t[1] = l4[1], t[2] = l4[2], t[3] = l4[3];
    t[4] = h4[0], t[5] = h4[1], t[6] = h4[2], t[7] = h4[3];
    return t;
  };

  constexpr int NK = 2 * KSTEPS;  // K fragments per tile
  constexpr int NV = 4 * DBLK;    // V^T fragments per tile
  // Fragments in flight.  Mode 4 holds a K and a V tile's bytes in registers across the iteration
  // and keeps the rings short: with 6 and 4 it spills 17 registers at two workgroups per CU (head
  // size 128), with 4 and 2 none, and the second workgroup is worth 224 -> 136 us on a pass of
  // four 512-token chunks over 2048 cached tokens.
  constexpr int KPRE = MODE == 4 ? 4 : 6;  // K fragments
  constexpr int VPRE = MODE == 4 ? 2 : 4;  // V^T fragments

  const int last_tile = ntiles - 1;
  // Block-table entries are vector loads (the load-to-LDS instruction is opaque to the
  // compiler, so it cannot prove the table unchanged and scalar), and waiting for one means
  // waiting for every tile load in flight.  So the entries of tile t + 3 are requested right
  // behind the loads issued in iteration t and read after the barrier of iteration t + 1, where
  // everything in flight has landed anyway; K(t + 2) and, one iteration later, V(t + 2) use them.
  struct Requested {
    int raw[NLK > 0 ? NLK : 1];
  };
  auto request = [&](int kt) {
    Requested r = {};
    if constexpr (NLK > 0) {
      const int t = min(kt, last_tile);  // past the end: any valid entry, never used
#pragma unroll
      for (int j = 0; j < NLK; ++j) r.raw[j] = a.pt[(int64_t)b * a.pt_rs + div_block(a, lookup_key(t, j))];
    }
    return r;
  };
  auto resolve = [&](const Requested &r) {
    Blocks blk = {};
    if constexpr (NLK > 0) {
#pragma unroll
      for (int j = 0; j < NLK; ++j) {
        const int p = MODE == 4 ? r.raw[j] : __builtin_amdgcn_readfirstlane(r.raw[j]);  // mode 4: per lane
        blk.phys[j] = (unsigned)p >= (unsigned)a.nb ? 0 : p;
      }
    }
    return blk;
  };
  auto kbuf = [&](int t) { return t & 1; };
  auto vbuf = [&](int t) { return t & 1; };
  int kt_begin = first_tile;
  Blocks blk_v = resolve(request(first_tile));     // blocks of the tile whose V is loaded next
  Blocks blk_k = resolve(request(first_tile + 1));  // ... whose K is loaded next
  Requested req = request(first_tile + 2);
  if constexpr (MODE == 4) {
    commit_bfp8(fetch_bfp8(a.k, first_tile, blk_v), false, first_tile & 1);
    commit_bfp8(fetch_bfp8(a.v, first_tile, blk_v), true, first_tile & 1);
    if (last_tile >= first_tile + 1)
      commit_bfp8(fetch_bfp8(a.k, first_tile + 1, blk_k), false, (first_tile + 1) & 1);
  } else {
    issue(a.k, ld_k, false, first_tile, kbuf(first_tile), blk_v);
    issue(a.v, ld_v, true, first_tile, vbuf(first_tile), blk_v);
    if (last_tile >= first_tile + 1) issue(a.k, ld_k, false, first_tile + 1, kbuf(first_tile + 1), blk_k);
  }
  blk_v = blk_k;
  wait_loads_and_sync();
  // The first K fragments of a tile are read one tile ahead (K(t+1) has landed at the barrier
  // of tile t), so the score product starts without waiting for LDS.
  bf16x8 ring[KPRE];
  if (wave_active && kt_begin < ntiles) {
#pragma unroll
    for (int i = 0; i < KPRE; ++i) ring[i] = read_k(smem + (kt_begin & 1) * T::STAGE_BYTES, i);
  }
  for (int kt = kt_begin; kt < ntiles; ++kt) {
    const unsigned char *cur = smem + (kt & 1) * T::STAGE_BYTES;
    const int key0 = kt * kKeysPerTile;
    // wavefront-uniform; with a window, tiles wholly below this wavefront's rows are skipped
    const bool compute = wave_active && key0 <= wave_last_key && key0 + kKeysPerTile > wave_first_key;

    // ---- S^T = K . Q^T -------------------------------------------------------------------
    floatx16 st[RH][2];
    if (compute) {
#pragma unroll
      for (int x = 0; x < RH; ++x)
#pragma unroll
        for (int r = 0; r < 16; ++r) st[x][0][r] = 0.f, st[x][1][r] = 0.f;
#pragma unroll
      for (int i = 0; i < NK; ++i) {
#pragma unroll
        for (int x = 0; x < RH; ++x)
          st[x][i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i % KPRE], qf[x][i >> 1], st[x][i & 1], 0, 0, 0);
        if (i + KPRE < NK) ring[i % KPRE] = read_k(cur, i + KPRE);
      }
      // pin the order: one fragment read behind the matrix instructions that use a fragment
#pragma unroll
      for (int i = 0; i < NK; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, RH, 0);
        if (i + KPRE < NK) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
    // K(kt+1) and V(kt) have landed for everyone; everyone is done with K(kt) and V(kt-1)
    wait_loads_and_sync();
    blk_k = resolve(req);  // blocks of tile kt + 2; blk_v holds those of tile kt + 1
    Staged k_staged = {}, v_staged = {};
    if constexpr (MODE == 4) {
      if (kt + 2 <= last_tile) k_staged = fetch_bfp8(a.k, kt + 2, blk_k);
      if (kt + 1 <= last_tile) v_staged = fetch_bfp8(a.v, kt + 1, blk_v);
    } else {
      if (kt + 2 <= last_tile) issue(a.k, ld_k, false, kt + 2, kt & 1, blk_k);
      if (kt + 1 <= last_tile) issue(a.v, ld_v, true, kt + 1, (kt + 1) & 1, blk_v);
    }
    blk_v = blk_k;
    req = request(kt + 3);

    if (compute) {
      bf16x8 vring[VPRE];
#pragma unroll
      for (int j = 0; j < VPRE; ++j) vring[j] = read_v(cur + T::TILE_BYTES, j);

      // ---- mask, online softmax (one query row per lane and row block) ----------------------
      // The softmax scale is positive, so the running maximum is tracked on raw scores and
      // the scale is folded into the exponent: p = exp2(s * c - m * c).
      const bool need_mask = (a.causal && key0 + kKeysPerTile - 1 > offset + row0) ||
                             key0 + kKeysPerTile > a.skv || a.mask != nullptr ||
                             (a.window > 0 && key0 <= offset + row0 + ROWS - 1 - a.window);
      bf16x8 pf[RH][4];
#pragma unroll
      for (int x = 0; x < RH; ++x) {
        const int qrow = row0 + 32 * x + n;
        if (need_mask) {  // wavefront-uniform: only diagonal / ragged / window-edge / explicitly masked tiles
          const int limit = a.causal ? min(offset + qrow, a.skv - 1) : a.skv - 1;
          const int lowest = a.window > 0 ? offset + qrow - a.window + 1 : 0;
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int key = key0 + 32 * kb + 8 * (r >> 2) + 4 * h + (r & 3);
              float v = st[x][kb][r];
              if (a.mask) {
                const int kc = min(key, a.skv - 1), qc = min(qrow, a.sq - 1);
                // additive mask is in natural-log units of the scaled score
                v += bf16_lo(a.mask[b * a.mask_bs + (int64_t)qc * a.mask_rs + kc]) *
                     (1.4426950408889634f / a.scale_log2e);
              }
              st[x][kb][r] = (key > limit || key < lowest) ? -INFINITY : v;
            }
        }
        // The first maximum is an ordinary compiler-visible read of both score blocks.
        float mloc = fmaxf(st[x][0][0], st[x][1][0]);
#pragma unroll
        for (int r = 1; r < 16; r += 3) {
          mloc = max3(mloc, st[x][0][r], st[x][1][r]);
          mloc = max3(mloc, st[x][0][r + 1], st[x][1][r + 1]);
          mloc = max3(mloc, st[x][0][r + 2], st[x][1][r + 2]);
        }
        {  // The other half of the key rows sits 32 lanes away.  v_permlane32_swap exchanges the
           // upper 32 lanes of its first operand with the lower 32 of its second; with two copies
           // of the value each lane ends up holding its own and its partner's.  Written as
           // assembly: through the builtin the compiler folds the two results into one.
          float ma = mloc, mb = mloc;
          asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(ma), "+v"(mb));
          mloc = max3(ma, mb, mb);
        }
        // Lazy rescaling: the running maximum only moves when a row's new maximum exceeds it
        // by more than 2^8 in the exponent domain.  Until then probabilities are taken
        // relative to the stale maximum (they may reach 2^8, harmless in bf16 / fp32), the
        // accumulators need no rescale, and the final division by the row sum is unchanged.
        const float kLazy = 8.0f;
        const bool move = !((mloc - m_run[x]) * a.scale_log2e <= kLazy);  // also true from -inf
        const float m_new = move ? mloc : m_run[x];
        const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = move ? __builtin_amdgcn_exp2f((m_run[x] - m_safe) * a.scale_log2e) : 1.0f;
        const float mc = m_safe * a.scale_log2e;
        m_run[x] = m_new;
        // skip the accumulator rescale when no row of the block moved its maximum
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
          for (int i = 0; i < DBLK; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[x][i][r] *= alpha;
        }
        // Probabilities as bf16 B-operand fragments: element e of key step k4 = 2 kb + s is
        // accumulator register 8 s + e of score block kb.  The row sum is taken over the rounded
        // values (two per v_dot2_f32_bf16), i.e. over exactly what the second product sees.
        const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
        float lsum = 0.f;
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            const int r = 8 * (k4 & 1) + e;
            const float p0 = __builtin_amdgcn_exp2f(fmaf(st[x][k4 >> 1][r], a.scale_log2e, -mc));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(st[x][k4 >> 1][r + 1], a.scale_log2e, -mc));
            const bf16x2 pp = {(__bf16)p0, (__bf16)p1};
            pf[x][k4][e] = pp[0], pf[x][k4][e + 1] = pp[1];
            lsum = __builtin_amdgcn_fdot2_f32_bf16(pp, ones, lsum, false);
          }
        l_run[x] = l_run[x] * alpha + lsum;
      }

      // ---- O^T += V^T . P^T -----------------------------------------------------------------
#pragma unroll
      for (int j = 0; j < NV; ++j) {
#pragma unroll
        for (int x = 0; x < RH; ++x)
          acc[x][j % DBLK] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vring[j % VPRE], pf[x][j / DBLK],
                                                                     acc[x][j % DBLK], 0, 0, 0);
        if (j + VPRE < NV) vring[j % VPRE] = read_v(cur + T::TILE_BYTES, j + VPRE);
      }
    }
    if constexpr (MODE == 4) {
      // K(kt+2) takes the place of K(kt), V(kt+1) that of V(kt-1): nobody reads either any more
      // (the barrier above), and the next barrier publishes what is written here
      if (kt + 2 <= last_tile) commit_bfp8(k_staged, false, kt & 1);
      if (kt + 1 <= last_tile) commit_bfp8(v_staged, true, (kt + 1) & 1);
    }
    if (wave_active && kt + 1 < ntiles && key0 + kKeysPerTile <= wave_last_key &&
        key0 + 2 * kKeysPerTile > wave_first_key) {  // this wavefront computes tile kt + 1
      const unsigned char *nxt = smem + ((kt + 1) & 1) * T::STAGE_BYTES;
#pragma unroll
      for (int i = 0; i < KPRE; ++i) ring[i] = read_k(nxt, i);
    }
  }

  // ---- normalise and store: lane (n, h) holds head-dim elements 32 db + 8 j + 4 h + i ----
  if constexpr (SPLIT) {
    if (!whole && wave_active) {
      // a part's accumulators and (maximum, sum) per row: lane l's four elements of group 4 db + j at float 256 (4 db + j) + 4 l
      // of the row block's, 1 KiB per store of the wavefront.  A row that sees none of the part's keys has maximum -inf, sum 0.
      const float l_tot = l_run[0] + __shfl_xor(l_run[0], 32);
      const PartLayout lay = part_layout(a);
      const int64_t at = (((int64_t)part * a.batch + b) * a.hq + hq) * lay.row_blocks + qt * RPW + wave / HPW;
      float *dst = a.part_acc + at * part_acc_floats(D) + 4 * lane;
#pragma unroll
      for (int db = 0; db < DBLK; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *reinterpret_cast<float4 *>(dst + 256 * (4 * db + j)) =
              make_float4(acc[0][db][4 * j], acc[0][db][4 * j + 1], acc[0][db][4 * j + 2], acc[0][db][4 * j + 3]);
      if (h == 0)
        *reinterpret_cast<float2 *>(a.part_acc + lay.slots * part_acc_floats(D) + at * (2 * kRowsPerWave) + 2 * n) =
            make_float2(m_run[0] * a.scale_log2e, l_tot);
      return;
    }
  }
  if (!wave_active) return;
#pragma unroll
  for (int x = 0; x < RH; ++x) {
    const float l_tot = l_run[x] + __shfl_xor(l_run[x], 32);
    const float inv = 1.0f / l_tot;
    const int qrow = row0 + 32 * x + n;
    if (qrow >= a.sq) continue;
    uint16_t *op = a.out + b * a.out_bs + hq * a.out_hs + (int64_t)qrow * a.out_ts + 4 * h;
#pragma unroll
    for (int db = 0; db < DBLK; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t lo = f32_to_bf16_bits(acc[x][db][4 * j] * inv) |
                      (f32_to_bf16_bits(acc[x][db][4 * j + 1] * inv) << 16);
        uint32_t hi = f32_to_bf16_bits(acc[x][db][4 * j + 2] * inv) |
                      (f32_to_bf16_bits(acc[x][db][4 * j + 3] * inv) << 16);
        *reinterpret_cast<uint2 *>(op + 32 * db + 8 * j) = make_uint2(lo, hi);
      }
  }
}

template <int D, int HPW, int MODE, bool SPLIT>
int launch_split(PrefillArgs &b, int grid, hipStream_t st) {
  const size_t lds = 2 * Tile<D>::STAGE_BYTES;  // two stages of a K and a V tile
  static std::atomic<uint64_t> lds_ready{0};
  if (!ensure_dynamic_lds(reinterpret_cast<const void *>(&prefill_kernel<D, HPW, MODE, SPLIT>), lds, lds_ready))
    return fail(TTPA_ERR_LAUNCH, "prefill: cannot reserve %zu bytes of LDS", lds);
  launch_dominant(&prefill_kernel<D, HPW, MODE, SPLIT>, dim3(grid, b.parts), dim3(256), lds, st, b);
  return check_launch("sdpa_prefill");
}

template <int D, int HPW, int MODE>
int launch_mode(const PrefillArgs &a, hipStream_t st) {
  PrefillArgs b = a;
  int grid = lay_out(b, HPW);
  b.parts = 1;
  if constexpr (MODE != 0) {
    constexpr SplitRule kRule = plain_split(D, MODE == 4);
    if (plain_splits(a) && a.part_acc && a.part_bytes >= part_bytes(a, HPW, kRule, D)) set_parts(b, HPW, kRule);
    if (b.parts > 1) {
      if (const int rc = launch_split<D, HPW, MODE, true>(b, grid, st)) return rc;
      prefill_merge_kernel<D><<<dim3((b.sq + kRowsPerWave - 1) / kRowsPerWave, b.hq, b.batch), dim3(2 * D), 0, st>>>(b);
      return check_launch("sdpa_prefill (merge of the parts)");
    }
  }
  if (MODE == 0 && a.fill_kc) grid = grid_with_fill(b, grid, D);
  return launch_split<D, HPW, MODE, false>(b, grid, st);
}

template <int D, int HPW>
int launch_bf16(const PrefillArgs &a, hipStream_t st) {
  if (stream_serves(a, D)) return launch_stream(a, D, st);
  if (!a.pt) return launch_mode<D, HPW, 0>(a, st);
  if (a.bs % kKeysPerTile == 0) return launch_mode<D, HPW, 1>(a, st);
  if (a.bs % Tile<D>::RPI == 0) return launch_mode<D, HPW, 3>(a, st);
  return launch_mode<D, HPW, 2>(a, st);
}

template <int D, int HPW>
int launch(const PrefillArgs &a, hipStream_t st) {
  if (a.pt && a.kv_bfp8) {
    // With scratch from the caller, a pass that the hand-scheduled loop can serve reads bfloat16
    // copies of its blocks (written by one launch in front of it) instead of expanding every
    // tile once per workgroup on its way into LDS.
    if (a.expand) {
      const int64_t blocks = (int64_t)a.batch * a.w;
      const int64_t cache_elems = blocks * a.hkv * a.bs * D;
      ExpandArgs e;
      e.kc = reinterpret_cast<const uint8_t *>(a.k), e.vc = reinterpret_cast<const uint8_t *>(a.v);
      e.k = static_cast<uint16_t *>(a.expand), e.v = e.k + cache_elems;
      e.table = reinterpret_cast<int32_t *>(e.v + cache_elems);
      e.pt = a.pt, e.pt_rs = a.pt_rs, e.chunk_start = a.chunk_start;
      e.batch = a.batch, e.w = a.w, e.hkv = a.hkv, e.bs = a.bs, e.nb = a.nb, e.sq = a.sq, e.causal = a.causal;
      e.by_pieces = divisor(a.bs * D / 1024), e.by_slabs = divisor(2 * a.hkv);  // (blocks are multiples of 32 tokens: stream_serves)
      // armed events: the pair brackets both launches
      hipEvent_t before, after;
      take_profile_events(before, after);
      const dim3 grid((unsigned)std::min<int64_t>((blocks * 2 * a.hkv * e.by_pieces.d + 3) / 4, kExpandWorkgroups));
      if (before)
        hipExtLaunchKernelGGL(bfp8_expand_kernel<D>, grid, dim3(256), 0u, st, before, nullptr, 0u, e);
      else
        bfp8_expand_kernel<D><<<grid, dim3(256), 0, st>>>(e);
      if (const int rc = check_launch("sdpa_prefill (block-float-8 expansion)")) return rc;
      if (after) arm_profile_events(nullptr, after);
      PrefillArgs b = a;
      b.k = e.k, b.v = e.v, b.pt = e.table, b.pt_rs = a.w, b.nb = (int)blocks, b.kv_bfp8 = 0, b.expand = nullptr;
      return launch_stream(b, D, st);
    }
    return launch_mode<D, HPW, 4>(a, st);
  }
  return launch_bf16<D, HPW>(a, st);
}

template <int D>
int launch_d(const PrefillArgs &a, hipStream_t st) {
  const int g = a.hq / a.hkv;
  if (g % 4 == 0) return launch<D, 4>(a, st);
  if (g % 2 == 0) return launch<D, 2>(a, st);
  return launch<D, 1>(a, st);
}

}  // namespace
}  // namespace ttpa

using namespace ttpa;

static int cus_for_rules() {
  const int cus = device_cus();
  return cus > 0 ? cus : 256;
}

// The cache fill that a dense prefill may carry along (ttpa_sdpa_prefill_fill).
struct FillSpec {
  void *k_cache, *v_cache;
  const int32_t *pt;
  int64_t pt_rs;
  const void *bidx;
  int bidx_i64, table_rows;
};

static int prefill_impl(void *out, int64_t out_batch_stride, int64_t out_head_stride,
                                 int64_t out_token_stride, const void *q, int64_t q_batch_stride,
                                 int64_t q_head_stride, int64_t q_token_stride, const void *k,
                                 const void *v, int64_t kv_batch_stride, int64_t kv_head_stride,
                                 int64_t kv_token_stride, const int32_t *page_table,
                                 int64_t page_table_row_stride, const int32_t *chunk_start,
                                 const void *mask, int64_t mask_batch_stride,
                                 int64_t mask_row_stride, int32_t batch, int32_t q_heads,
                                 int32_t kv_heads, int32_t q_len, int32_t kv_len, int32_t head_size,
                                 int32_t block_size, int32_t table_width, int32_t num_blocks,
                                 int32_t causal, float scale, int32_t sliding_window, void *stream,
                                 const FillSpec *fill = nullptr, int32_t kv_format = TTPA_KV_BF16,
                                 void *workspace = nullptr, int64_t workspace_bytes = 0, int64_t most_keys = 0) {
  TTPA_REQUIRE(out && q && k && v, "null pointer argument");
  TTPA_REQUIRE(sliding_window >= 0, "prefill: sliding_window %d is negative", sliding_window);
  TTPA_REQUIRE(sliding_window == 0 || causal, "prefill: a sliding window needs causal masking");
  TTPA_REQUIRE(batch > 0 && q_heads > 0 && kv_heads > 0 && q_len > 0 && head_size > 0,
               "non-positive dimension");
  TTPA_REQUIRE(q_heads % kv_heads == 0, "q_heads %d not divisible by kv_heads %d", q_heads,
               kv_heads);
  if (head_size != 64 && head_size != 128 && head_size != 256)
    return fail(TTPA_ERR_UNSUPPORTED, "prefill: head_size %d; supported 64, 128, 256", head_size);
  TTPA_REQUIRE(!(mask && causal), "an additive mask excludes causal masking");
  // the running maximum is tracked on raw scores and the mask is brought to their units by a
  // division: both need a positive scale
  TTPA_REQUIRE(scale > 0.f, "prefill: scale %g must be positive", (double)scale);
  if (page_table) {
    TTPA_REQUIRE(block_size > 0 && table_width > 0 && num_blocks > 0,
                 "paged form needs block_size, table_width and num_blocks");
    kv_len = table_width * block_size;
    TTPA_REQUIRE((int64_t)kv_len * block_size < (1ll << 32), "prefill: table_width * block_size^2 must stay below 2^32");
  } else {
    TTPA_REQUIRE(kv_len > 0, "dense form needs kv_len > 0");
    TTPA_REQUIRE(kv_batch_stride % 8 == 0 && kv_head_stride % 8 == 0 && kv_token_stride % 8 == 0,
                 "prefill: k / v strides must be multiples of 8 elements");
    // (both loops reach a tile's rows by unsigned 32-bit numbers of bytes from the first)
    TTPA_REQUIRE(kv_len == 1 || (kv_token_stride >= 0 && kv_token_stride < (1ll << 31) &&
                                 (std::min(kv_len, 64) - 1) * kv_token_stride < (1ll << 31) - 1024),
                 "prefill: k / v token stride %lld is negative, or a tile of 64 rows reaches over 4 GiB", (long long)kv_token_stride);
    TTPA_REQUIRE(chunk_start == nullptr, "chunk_start applies to the paged form only");
  }
  TTPA_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out),
               "prefill: q / k / v / out must be 16-byte aligned");
  TTPA_REQUIRE(q_batch_stride % 8 == 0 && q_head_stride % 8 == 0 && q_token_stride % 8 == 0 &&
                   out_batch_stride % 4 == 0 && out_head_stride % 4 == 0 && out_token_stride % 4 == 0,
               "prefill: q strides must be multiples of 8 elements, out strides of 4");
  TTPA_REQUIRE((int64_t)batch * q_heads * ((q_len + 31) / 32) < (1ll << 30),
               "prefill: batch * heads * query tiles too large for one launch");

  PrefillArgs a;
  a.out = static_cast<uint16_t *>(out);
  a.out_bs = out_batch_stride, a.out_hs = out_head_stride, a.out_ts = out_token_stride;
  a.q = static_cast<const uint16_t *>(q);
  a.q_bs = q_batch_stride, a.q_hs = q_head_stride, a.q_ts = q_token_stride;
  a.k = static_cast<const uint16_t *>(k);
  a.v = static_cast<const uint16_t *>(v);
  a.kv_bs = kv_batch_stride, a.kv_hs = kv_head_stride, a.kv_ts = kv_token_stride;
  a.pt = page_table, a.pt_rs = page_table_row_stride;
  a.chunk_start = chunk_start;
  a.mask = static_cast<const uint16_t *>(mask);
  a.mask_bs = mask_batch_stride, a.mask_rs = mask_row_stride;
  a.batch = batch, a.hq = q_heads, a.hkv = kv_heads, a.sq = q_len, a.skv = kv_len;
  a.bs = block_size, a.w = table_width, a.nb = num_blocks, a.causal = causal ? 1 : 0;
  a.cus = cus_for_rules();
  a.keys_known = page_table && most_keys > 0, a.keys_bound = a.keys_known ? std::min<int64_t>(most_keys, kv_len) : kv_len;
  a.window = sliding_window;
  a.scale_log2e = scale * 1.4426950408889634f;
  {
    // (TTPA_PREFILL_STREAM=0, read on every call, sends every shape through the plain loop)
    const char *e = getenv("TTPA_PREFILL_STREAM");
    a.stream = e ? atoi(e) : 1;
  }
  if (kv_format != TTPA_KV_BF16 && kv_format != TTPA_KV_BFP8)
    return fail(TTPA_ERR_INVALID_ARGUMENT, "prefill: unknown kv_format %d", kv_format);
  a.kv_bfp8 = kv_format == TTPA_KV_BFP8;
  a.expand = nullptr;
  if (a.kv_bfp8) {
    TTPA_REQUIRE(page_table != nullptr, "prefill: a block-float-8 K / V is a paged cache");
    if (block_size % 16)
      return fail(TTPA_ERR_UNSUPPORTED, "prefill: a block-float-8 cache needs block_size %% 16 == 0");
    TTPA_REQUIRE(workspace_bytes >= 0 && (workspace != nullptr || workspace_bytes == 0),
                 "prefill: workspace_bytes %lld with a null workspace", (long long)workspace_bytes);
    const int64_t need = expand_bytes(batch, table_width, kv_heads, block_size, head_size);
    if (stream_expands(a, head_size, workspace_bytes) && workspace && aligned16(workspace) && (int64_t)batch * table_width < (1ll << 31) && workspace_bytes >= need) {
      a.expand = workspace;  // (a smaller one is not an error: the pass expands tile by tile instead)
      workspace = static_cast<unsigned char *>(workspace) + need;
      workspace_bytes -= need;
    }
  }
  a.part_acc = nullptr, a.part_bytes = 0, a.parts = 1;
  if (page_table && workspace && aligned16(workspace)) a.part_acc = static_cast<float *>(workspace), a.part_bytes = workspace_bytes;
  a.bs_magic = block_size >= 2 ? (uint32_t)((1ull << 32) / (uint32_t)block_size) + 1u : 0u;
  a.fill_kc = a.fill_vc = nullptr;
  a.fill_pt = nullptr, a.fill_pt_rs = 0, a.fill_bidx = nullptr, a.fill_bidx_i64 = 0, a.fill_rows = 0;
  a.fill_groups = a.attn_per_fill = a.n_fill = 0;
  if (fill) {
    a.fill_kc = static_cast<uint16_t *>(fill->k_cache), a.fill_vc = static_cast<uint16_t *>(fill->v_cache);
    a.fill_pt = fill->pt, a.fill_pt_rs = fill->pt_rs;
    a.fill_bidx = fill->bidx, a.fill_bidx_i64 = fill->bidx_i64, a.fill_rows = fill->table_rows;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (head_size) {
    case 64: return launch_d<64>(a, st);
    case 128: return launch_d<128>(a, st);
    default: return launch_d<256>(a, st);
  }
}

#define TTPA_PREFILL_PARAMS                                                                        \
  void *out, int64_t out_batch_stride, int64_t out_head_stride, int64_t out_token_stride,          \
      const void *q, int64_t q_batch_stride, int64_t q_head_stride, int64_t q_token_stride,        \
      const void *k, const void *v, int64_t kv_batch_stride, int64_t kv_head_stride,               \
      int64_t kv_token_stride, const int32_t *page_table, int64_t page_table_row_stride,           \
      const int32_t *chunk_start, const void *mask, int64_t mask_batch_stride,                     \
      int64_t mask_row_stride, int32_t batch, int32_t q_heads, int32_t kv_heads, int32_t q_len,    \
      int32_t kv_len, int32_t head_size, int32_t block_size, int32_t table_width,                  \
      int32_t num_blocks, int32_t causal, float scale
#define TTPA_PREFILL_ARGS                                                                          \
  out, out_batch_stride, out_head_stride, out_token_stride, q, q_batch_stride, q_head_stride,      \
      q_token_stride, k, v, kv_batch_stride, kv_head_stride, kv_token_stride, page_table,          \
      page_table_row_stride, chunk_start, mask, mask_batch_stride, mask_row_stride, batch,         \
      q_heads, kv_heads, q_len, kv_len, head_size, block_size, table_width, num_blocks, causal,    \
      scale

extern "C" int ttpa_sdpa_prefill(TTPA_PREFILL_PARAMS, void *stream) {
  return prefill_impl(TTPA_PREFILL_ARGS, 0, stream);
}

extern "C" int ttpa_sdpa_prefill_windowed(TTPA_PREFILL_PARAMS, int32_t sliding_window, void *stream) {
  return prefill_impl(TTPA_PREFILL_ARGS, sliding_window, stream);
}

extern "C" int ttpa_sdpa_prefill_format(TTPA_PREFILL_PARAMS, int32_t sliding_window, int32_t kv_format,
                                        void *stream) {
  return prefill_impl(TTPA_PREFILL_ARGS, sliding_window, stream, nullptr, kv_format);
}

extern "C" int ttpa_sdpa_prefill_expanded(TTPA_PREFILL_PARAMS, int32_t sliding_window, int32_t kv_format,
                                          void *workspace, int64_t workspace_bytes, void *stream) {
  return prefill_impl(TTPA_PREFILL_ARGS, sliding_window, stream, nullptr, kv_format, workspace, workspace_bytes);
}

extern "C" int ttpa_sdpa_prefill_bounded(TTPA_PREFILL_PARAMS, int32_t sliding_window, int32_t kv_format, int64_t most_keys,
                                         void *workspace, int64_t workspace_bytes, void *stream) {
  return prefill_impl(TTPA_PREFILL_ARGS, sliding_window, stream, nullptr, kv_format, workspace, workspace_bytes, most_keys);
}

extern "C" int64_t ttpa_sdpa_prefill_workspace_bytes(int32_t batch, int32_t kv_heads, int32_t head_size,
                                                     int32_t block_size, int32_t table_width, int32_t kv_format) {
  if (kv_format != TTPA_KV_BFP8 || batch <= 0 || kv_heads <= 0 || head_size <= 0 || block_size <= 0 || table_width <= 0)
    return 0;
  return expand_bytes(batch, table_width, kv_heads, block_size, head_size);
}

extern "C" int64_t ttpa_sdpa_prefill_scratch_bytes(int32_t batch, int32_t q_heads, int32_t kv_heads, int32_t q_len, int32_t head_size,
                                                   int32_t block_size, int32_t table_width, int32_t kv_format) {
  return ttpa_sdpa_prefill_bounded_scratch_bytes(batch, q_heads, kv_heads, q_len, head_size, block_size, table_width, kv_format, 0);
}

extern "C" int64_t ttpa_sdpa_prefill_bounded_scratch_bytes(int32_t batch, int32_t q_heads, int32_t kv_heads, int32_t q_len,
                                                           int32_t head_size, int32_t block_size, int32_t table_width,
                                                           int32_t kv_format, int64_t most_keys) {
  if (batch <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads || q_len <= 0 || head_size <= 0 || block_size <= 0 || table_width <= 0)
    return 0;
  const int32_t some_table = 0;
  PrefillArgs a = {};
  a.pt = &some_table, a.stream = 1, a.cus = cus_for_rules();
  a.batch = batch, a.hq = q_heads, a.hkv = kv_heads, a.sq = q_len, a.bs = block_size, a.w = table_width;
  a.keys_bound = (int64_t)table_width * block_size;
  if (most_keys > 0) a.keys_known = 1, a.keys_bound = std::min(a.keys_bound, most_keys);
  if (kv_format == TTPA_KV_BFP8) {
    if (!stream_expands(a, head_size, INT64_MAX)) return plain_part_bytes(a, head_size, true);
    return ttpa_sdpa_prefill_workspace_bytes(batch, kv_heads, head_size, block_size, table_width, kv_format) + stream_part_bytes(a, head_size);
  }
  return stream_serves(a, head_size) ? stream_part_bytes(a, head_size) : plain_part_bytes(a, head_size, false);
}

extern "C" int ttpa_sdpa_prefill_fill(
    void *out, int64_t out_batch_stride, int64_t out_head_stride, int64_t out_token_stride,
    const void *q, int64_t q_batch_stride, int64_t q_head_stride, int64_t q_token_stride,
    const void *k, const void *v, int64_t kv_batch_stride, int64_t kv_head_stride,
    int64_t kv_token_stride, int32_t batch, int32_t q_heads, int32_t kv_heads, int32_t q_len,
    int32_t kv_len, int32_t head_size, int32_t causal, float scale, int32_t sliding_window,
    void *k_cache, void *v_cache, const int32_t *fill_page_table, int64_t fill_page_table_row_stride,
    const void *batch_idx, int batch_idx_is_i64, int32_t table_rows, int32_t block_size,
    int32_t table_width, int32_t num_blocks, void *stream) {
  TTPA_REQUIRE(k_cache && v_cache && fill_page_table, "prefill + fill: null cache / page_table pointer");
  TTPA_REQUIRE(block_size > 0 && table_width > 0 && num_blocks > 0 && table_rows > 0,
               "prefill + fill: non-positive cache geometry");
  TTPA_REQUIRE(batch_idx != nullptr || batch <= 1, "batch_idx may only be omitted for a single-user fill");
  TTPA_REQUIRE((int64_t)kv_len <= (int64_t)table_width * block_size,
               "kv_len %d does not fit %d page-table columns of %d tokens", kv_len, table_width, block_size);
  TTPA_REQUIRE((int64_t)kv_len * block_size < (1ll << 32), "prefill + fill: kv_len * block_size must stay below 2^32");
  TTPA_REQUIRE(aligned16(k_cache) && aligned16(v_cache), "prefill + fill: caches must be 16-byte aligned");
  const FillSpec fill{k_cache, v_cache, fill_page_table, fill_page_table_row_stride, batch_idx,
                      batch_idx_is_i64, table_rows};
  return prefill_impl(out, out_batch_stride, out_head_stride, out_token_stride, q, q_batch_stride,
                      q_head_stride, q_token_stride, k, v, kv_batch_stride, kv_head_stride,
                      kv_token_stride, nullptr, 0, nullptr, nullptr, 0, 0, batch, q_heads, kv_heads,
                      q_len, kv_len, head_size, block_size, table_width, num_blocks, causal, scale,
                      sliding_window, stream, &fill);
}

extern "C" int ttpa_split_key_prefill(
    void *out, int64_t out_batch_stride, int64_t out_head_stride, int64_t out_token_stride, const void *q_nope,
    int64_t q_nope_batch_stride, int64_t q_nope_head_stride, int64_t q_nope_token_stride, const void *q_rope,
    int64_t q_rope_batch_stride, int64_t q_rope_head_stride, int64_t q_rope_token_stride, const void *k_nope,
    int64_t k_nope_batch_stride, int64_t k_nope_head_stride, int64_t k_nope_token_stride, const void *k_rope,
    int64_t k_rope_batch_stride, int64_t k_rope_head_stride, int64_t k_rope_token_stride, const void *v,
    int64_t v_batch_stride, int64_t v_head_stride, int64_t v_token_stride, int32_t batch, int32_t q_heads,
    int32_t kv_heads, int32_t seq_len, float scale, void *stream) {
  TTPA_REQUIRE(out && q_nope && q_rope && k_nope && k_rope && v, "null pointer argument");
  TTPA_REQUIRE(batch > 0 && q_heads > 0 && kv_heads > 0 && seq_len > 0, "non-positive dimension");
  TTPA_REQUIRE(q_heads % kv_heads == 0, "q_heads %d not divisible by kv_heads %d", q_heads, kv_heads);
  TTPA_REQUIRE(seq_len % 32 == 0, "split-key prefill: seq_len %d is not a multiple of 32", seq_len);
  TTPA_REQUIRE(scale > 0.f, "split-key prefill: scale %g must be positive", (double)scale);
  TTPA_REQUIRE(aligned16(out) && aligned16(q_nope) && aligned16(q_rope) && aligned16(k_nope) && aligned16(k_rope) && aligned16(v),
               "split-key prefill: operands must be 16-byte aligned");
  const int64_t strides[] = {q_nope_batch_stride, q_nope_head_stride, q_nope_token_stride, q_rope_batch_stride, q_rope_head_stride,
                             q_rope_token_stride, k_nope_batch_stride, k_nope_head_stride, k_nope_token_stride, k_rope_batch_stride,
                             k_rope_head_stride, k_rope_token_stride, v_batch_stride, v_head_stride, v_token_stride};
  for (int64_t s : strides) TTPA_REQUIRE(s % 8 == 0, "split-key prefill: operand strides must be multiples of 8 elements");
  TTPA_REQUIRE(out_batch_stride % 4 == 0 && out_head_stride % 4 == 0 && out_token_stride % 4 == 0,
               "split-key prefill: out strides must be multiples of 4 elements");
  // (but for the queries', token strides are unsigned 32-bit numbers of bytes in the kernel)
  TTPA_REQUIRE(k_nope_token_stride >= 0 && k_nope_token_stride < (1 << 24) && k_rope_token_stride >= 0 && k_rope_token_stride < (1 << 24) &&
                   v_token_stride >= 0 && v_token_stride < (1 << 24) && q_nope_token_stride < (1ll << 31) && out_token_stride >= 0 &&
                   out_token_stride < (1ll << 31),
               "split-key prefill: token stride out of range");
  TTPA_REQUIRE((int64_t)batch * q_heads * ((seq_len + 31) / 32) < (1ll << 30),
               "split-key prefill: batch * heads * query tiles too large for one launch");
  PrefillArgs a = {};
  a.out = static_cast<uint16_t *>(out);
  a.out_bs = out_batch_stride, a.out_hs = out_head_stride, a.out_ts = out_token_stride;
  a.q = static_cast<const uint16_t *>(q_nope);
  a.q_bs = q_nope_batch_stride, a.q_hs = q_nope_head_stride, a.q_ts = q_nope_token_stride;
  a.q2 = static_cast<const uint16_t *>(q_rope);
  a.q2_bs = q_rope_batch_stride, a.q2_hs = q_rope_head_stride, a.q2_ts = q_rope_token_stride;
  a.k = static_cast<const uint16_t *>(k_nope);
  a.kv_bs = k_nope_batch_stride, a.kv_hs = k_nope_head_stride, a.kv_ts = k_nope_token_stride;
  a.k2 = static_cast<const uint16_t *>(k_rope);
  a.k2_bs = k_rope_batch_stride, a.k2_hs = k_rope_head_stride, a.k2_ts = k_rope_token_stride;
  a.v = static_cast<const uint16_t *>(v);
  a.v_bs = v_batch_stride, a.v_hs = v_head_stride, a.v_ts = v_token_stride;
  a.batch = batch, a.hq = q_heads, a.hkv = kv_heads, a.sq = seq_len, a.skv = seq_len, a.causal = 1, a.parts = 1;
  a.scale_log2e = scale * 1.4426950408889634f;
  return launch_stream_wide(a, static_cast<hipStream_t>(stream));
}
