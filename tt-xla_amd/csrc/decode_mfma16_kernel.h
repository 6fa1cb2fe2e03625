// Paged decode attention on the 16x16x32 matrix-core shape: up to 16 query heads per KV head,
// 32 or 64 KiB of tiles in LDS per workgroup of four wavefronts, and 16 KiB of tables; head sizes 64, 128 and 256 with a block-float-8 cache (expanded
// to half precision) or a bfloat16 cache.
//
// Work decomposition, partial slots and merge kernel are those of decode.hip, with tiles of
// 64, 32 or 32 tokens at head size 64, 128, 256, or 64 at 128 (tile_bytes).  Inside a wavefront a tile of K,
// then of V, goes global -> registers -> a wave-private LDS buffer of that size that both
// tensors use in turn:
//   stage K(t) | prefetch K(t+1) | S^T = K Q^T | softmax | stage V(t) | prefetch V(t+1) | O^T += V^T P^T
// so every global load has three quarters of a tile period to arrive.  The byte -> half
// expansion of the block-float-8 cache is the one of decode_mfma.hip (one permute and one
// packed fma per element pair, exponents relative to the tile's largest, running reference
// exponent for the V accumulator).
//
// FUSED: the kernel also performs the decode step's cache update.  The token at cur_pos of a
// user sits in the last tile of each of its segments, and that tile belongs to exactly one
// wavefront: it takes the token's K / V rows from the fresh activations instead of the cache
// (quantising them for a block-float-8 cache) and stores them into the cache, so nobody
// depends on a separate update launch.  The fresh rows of a segment's (user, head) are
// requested where its Q rows are, once per segment (that block has its own waits; a request
// inside the per-tile path would make the wait-count pass drain the tile loads in the
// steady-state loop).  Users whose position is negative (padded rows) attend nothing; their write
// is the merge kernel's (write_negative_position).
//
// v_mfma_f32_16x16x32_{f16,bf16} with the heads as the 16-wide N dimension:
//   S^T block b (16 keys):  A = K rows 16 b + lane%16, 8 elements per lane and k-step
//                           B = Q, lane%16 = head;   C: lane (head, quad) holds keys 16 b + 4 quad + r
//   O^T block db (16 d):    the 32 k slots of a step are the keys lane (., quad) already holds
//                           from blocks 2 s and 2 s + 1, so the probabilities are the B operand
//                           as they are; A = V^T through two transposing LDS loads (4 keys each)
// Compared with the 32x32x16 kernel, a lane carries half the scores and half the
// accumulator, and the matrix pipe is busy half as long per tile.
//
// LDS tile: rows of 2 * head_size bytes, unpadded, 16-byte chunks stored at
// chunk ^ (row & 15) for K (A-operand reads: 16 rows, one chunk column) and at
// chunk ^ (2 y | y & 1), y = row & 7, for V (transposing reads: 32 lanes cover 8 rows x 2
// chunks); both make the staging writes of two neighbouring rows land in different banks too.
// (The exchange stays inside an aligned group of 16 chunks = 256 bytes = every bank once.)
// Head size 64: a row is half a bank period, so two neighbouring rows already differ in their
// banks and the keys are taken from row / 2: (row / 2) & 7 and y = (row / 2) & 3.
//
// Where a tile's rows sit in the cache (RUNS): one run of consecutive rows when a block holds
// whole tiles; two runs of half a tile when block_size is a multiple of half a tile (the serving
// default of 32 with head size 64, or with 128 and block-float-8; 16 with 256); four runs of a quarter
// tile when it is a multiple of a quarter tile (16 with 64; 8 with 128 and 256); otherwise
// one run per load instruction.  A run costs a block-table lookup and a 64-bit base, which are
// scalar registers, the resource this kernel is short of.
//
// This header holds the kernel and its launcher; one translation unit per head size
// instantiates it (decode_mfma16_d64.hip, _d128.hip, _d256.hip).
#pragma once
#include "decode_common.h"

namespace ttpa {
namespace decode {
namespace {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef short shortx4 __attribute__((ext_vector_type(4)));

constexpr int kMaxUsers16 = kMaxUsers;  // the library-wide limit: 16 KiB of prefix tables
// Bytes of a tile's K (or V) rows as 16-bit elements, i.e. of a wavefront's LDS buffer: 16 KiB
// (32 tokens) at head size 256, 8 KiB (64 / 32 tokens) at head size 64 / 128.  A wavefront has one
// tile of K and one of V in flight; the kernel ends when the slowest wavefront has drained its last tile, and wavefronts of one launch finish
// several microseconds apart (the XCDs do not get equal shares of the HBM bandwidth), so a
// shorter tile shortens that tail: config 2's step 58.7 -> 57.8 us, config 4's 549 -> 543 us.
// At head size 64 (64 / 8 heads, us per layer of a replayed step): a window of 1024 over 37 users 25.2 ->
// 23.1 (its two ends waste less, too), 32 users with 512 ... 4096 tokens 27.7 -> 26.5, 8 users with
// 128 ... 1024 15.0 -> 11.6, 128 users with 256 ... 32768 274 -> 272; 4 KiB: 23.6, 26.9, 10.8.
// A block-float-8 tile is half the bytes behind the same chain of steps, so that kernel is bound by the chain.  With 16 KiB (LONG) it
// needed 316 registers, one wavefront per SIMD; with 8 KiB two share a SIMD and a launch has twice the wavefronts (us per layer,
// 64 users with 1024 ... 16384 tokens, 32/8 heads at head size 128: 144 -> 137; 100 users with 1024 ... 8192, 64/8 heads at 64: 92 ->
// 78; 40 users of 16/16 heads with 512 ... 4096: 68 -> 61).  Wide groups keep 16 KiB (DecodeArgs::long_tiles).  Head size 256 has
// 32-token tiles either way.
template <int D, bool LONG = false>
constexpr int tile_bytes() {
  return D <= 128 && !LONG ? 8192 : 16384;
}

template <bool F16>
__device__ __forceinline__ floatx4 mma16(const u32x4 &x, const u32x4 &y, const floatx4 &c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, x),
                                                  __builtin_bit_cast(halfx8, y), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x),
                                                   __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
}

// A pair of non-negative bfloat16 values less `n` units of their last place each (0 stays 0, NaN stays NaN).
__device__ __forceinline__ uint32_t less_units(uint32_t pair, uint32_t n) {
  typedef uint16_t ushort2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(ushort2_t, pair), __builtin_bit_cast(ushort2_t, n)));
}

// The end of a segment that one workgroup of WAVES wavefronts has read (`active` of them had a tile): the
// wavefronts' results meet in LDS, each in its own tile buffer, whose last tile it has consumed; then every
// thread merges, normalises and stores four neighbouring elements of a head.  A wavefront's values lie as
// its lanes hold them, [element / 4][head][4], so its stores are 1 KiB in a row.
template <int D, int WAVES>
__device__ __forceinline__ void merge_waves(const DecodeArgs &a, int u, int h, int G, int active, uint8_t *own, const uint8_t *all,
                                            int pitch, const floatx4 (&acc)[D / 16], float vout, float m, float l) {
  __shared__ float s_m[WAVES][16], s_l[WAVES][16];
  const int lane = threadIdx.x & 63, wib = threadIdx.x >> 6;
  if (wib < active) {
#pragma unroll
    for (int db = 0; db < D / 16; ++db)
      *reinterpret_cast<float4 *>(own + db * 1024 + lane * 16) =
          make_float4(acc[db][0] * vout, acc[db][1] * vout, acc[db][2] * vout, acc[db][3] * vout);
    if (lane < 16) s_m[wib][lane] = m, s_l[wib][lane] = l;
  }
  __syncthreads();
  const int gshift = G <= 1 ? 0 : 32 - __builtin_clz(G - 1);
  const bool wide_stores = ((a.out_us | a.out_hs) & 3) == 0;
  for (int i = threadIdx.x; i < (D / 4) << gshift; i += kWave * WAVES) {
    const int g = i & ((1 << gshift) - 1), d4 = i >> gshift;
    if (g >= G) continue;
    float mall = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      if (w < active) mall = fmaxf(mall, s_m[w][g]);
    const float ref = merge_reference(mall);
    float num[4] = {0.f, 0.f, 0.f, 0.f}, den = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      if (w < active) {
        const float wgt = __builtin_amdgcn_exp2f(s_m[w][g] - ref);
        const float4 x = *reinterpret_cast<const float4 *>(all + w * pitch + d4 * 256 + g * 16);
        num[0] = fmaf(wgt, x.x, num[0]), num[1] = fmaf(wgt, x.y, num[1]);
        num[2] = fmaf(wgt, x.z, num[2]), num[3] = fmaf(wgt, x.w, num[3]);
        den = fmaf(wgt, s_l[w][g], den);
      }
    if (a.sink) {  // the sink logit (natural-log units, not scaled) only enlarges the normaliser
      const float sk = a.sink[h * G + g] * 1.4426950408889634f;
      const float mnew = fmaxf(mall, sk);
      const float resc = __builtin_amdgcn_exp2f(mall - mnew);
#pragma unroll
      for (int r = 0; r < 4; ++r) num[r] *= resc;
      den = den * resc + __builtin_amdgcn_exp2f(sk - mnew);
    }
    uint16_t *dst = a.out + u * a.out_us + (int64_t)(h * G + g) * a.out_hs + 4 * d4;
    uint32_t b[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) b[r] = f32_to_bf16_bits(num[r] / den);
    if (wide_stores) {
      *reinterpret_cast<uint2 *>(dst) = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[r] = (uint16_t)b[r];
    }
  }
}

// RUNS: 1, 2, 4, or 0 for one run per load.  MASKED: an additive mask row per (user, head) joins the
// scores (a.mask; the form of a pass that is not causal, built with RUNS = 0 and without the update).
// DIRECT: a workgroup of DIRECT wavefronts owns the whole segment blockIdx.x (chosen by direct_waves, decode.hip): no prefix, no
// search, no partials, no merge launch.  Its wavefronts take the segment's tiles in turn.  LONG: tiles of 16 KiB (a.long_tiles).
template <int D, bool BFP8, int RUNS, bool FUSED, bool MASKED = false, int DIRECT = 0, bool LONG = false, bool ONE = false>
// (Whole bfloat16 segments: no more than two wavefronts per SIMD, or the compiler saves registers for a third that has no segment: 37 users
// of 64/8 heads of 64 in a window of 1024 22.0 / 21.8 us per layer.  Block-float-8 ones use the third: 100 users of 64/8 of 64 19.4 / 16.5.)
__global__ __launch_bounds__(DIRECT ? kWave *DIRECT : 256) __attribute__((amdgpu_waves_per_eu((DIRECT || BFP8) && D <= 128 && !LONG ? 2 : 1, DIRECT && !BFP8 ? 2 : 8)))
void paged_decode_mfma16_kernel(
    DecodeArgs a, const int32_t *__restrict__ page_table, const void *__restrict__ cur_pos) {
  static_assert(D == 64 || D == 128 || D == 256, "shapes built");
  constexpr int kTileBytes = tile_bytes<D, LONG>();
  constexpr int TILE = kTileBytes / (2 * D);  // tokens per tile
  constexpr int ROWB = 2 * D;                 // bytes of a tile row in LDS
  constexpr int KSTEPS = D / 32, DBLK = D / 16;
  constexpr int KBLK = TILE / 16;     // score blocks (16 keys each) per tile
  constexpr int PSTEPS = TILE / 32;   // k-steps of the second product per tile
  // staging geometry: 16 bytes per lane, so a load instruction covers (head size 128) 8 whole
  // token rows of element bytes or 4 of bfloat16
  constexpr int BPE = BFP8 ? 1 : 2;   // bytes per cache element
  constexpr int LPR = D * BPE / 16;   // lanes per token row
  constexpr int RPL = 64 / LPR;       // rows per load
  constexpr int NL = TILE / RPL;      // loads per tile and tensor
  constexpr int GPR = D / 16;         // exponent bytes per row (block-float-8)
  constexpr int NOFF = RUNS == 0 ? NL : RUNS;  // runs of consecutive cache rows per tile
  constexpr int LPO = NL / NOFF;               // loads per run
  static_assert(NL % NOFF == 0, "a run is a whole number of loads");

  __shared__ int s_pref[DIRECT ? 1 : kMaxUsers16 + 1];
  __shared__ int s_len[DIRECT ? 1 : kMaxUsers16];
  __shared__ int s_wsum[kWavesPerBlock];
  extern __shared__ __attribute__((aligned(16))) uint8_t tiles[];

  int seg_units = 0, n_ranges = a.n_waves;
  if constexpr (DIRECT == 0) seg_units = build_prefix_units<TILE, BFP8 ? D <= 128 && !LONG : D == 256 && !MASKED && !ONE>(a, cur_pos, s_pref, s_len, s_wsum, n_ranges);
  const int lane = threadIdx.x & 63;
  const int wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, quad = lane >> 4;
  const int wave = blockIdx.x * kWavesPerBlock + wib;
  int64_t total = 0, x_lo = 0, x_hi = 0;
  int n_eff = 0, n_tiles = 0;
  Cursor cur;
  if constexpr (DIRECT > 0) {
    cur.u = (int)blockIdx.x / a.hkv;
    cur.h = (int)blockIdx.x - cur.u * a.hkv;
    n_tiles = tiles_of_user<TILE>(a, cur_pos, cur.u, cur.len);
    if (n_tiles == 0) {  // a padded row: NaN like softmax over nothing, and the parked token's cache write
      const int g_all = a.hq / a.hkv;
      for (int i = threadIdx.x; i < g_all * D; i += kWave * DIRECT)
        a.out[cur.u * a.out_us + (int64_t)(cur.h * g_all + i / D) * a.out_hs + i % D] = 0x7fc0;
      if constexpr (FUSED) write_negative_position(a, blockIdx.x, D);
      return;
    }
    cur.lo = window_lo(a, cur.len);
    cur.t = cur.lo / TILE + wib;
    cur.tiles_left = n_tiles - wib;
  } else {
    // The flat list in units: per segment `seg_units` units that stand for the cost of opening it,
    // then its tiles.  A range of more than seg_units units holds at least one tile.
    const int total_units = __builtin_amdgcn_readfirstlane(s_pref[a.users]);
    const Share share = share_of(total_units, a.hkv, n_ranges, seg_units, wave);
    total = share.total, n_eff = share.n_eff;
    if (total == 0 || wave >= n_eff) {
      publish_segment_row(a, s_pref, total, n_eff, seg_units);
      return;
    }
    x_lo = share.lo, x_hi = share.hi;
  }
  int64_t x = x_lo;  // set below to the unit of the first tile at or behind x_lo
  uint8_t *tile = tiles + wib * kTileBytes;
  const int G = ONE ? 1 : a.hq / a.hkv;

  // staging lane mapping and swizzled write positions
  const int sr = lane / LPR, sc = lane % LPR;
  const uint32_t lane_bytes = (uint32_t)(sr * D * BPE + sc * 16);
  // block-float-8: the lane's exponent byte (row sr, group sc) is fetched inside its aligned
  // dword and cut out when the tile is staged: a byte load is widened where it is issued, which
  // would make the loop wait for the next tile's exponents at the end of every iteration
  const uint32_t lane_exp = (uint32_t)((sr * GPR + sc) & ~3);
  const uint32_t exp_shift = (uint32_t)(8 * (sc & 3));
  const int64_t slab = BFP8 ? (int64_t)(a.bs + a.bs / 16) * D : (int64_t)a.bs * D * 2;  // bytes
  // A lane stages CPL chunks of 16 bytes (16-bit elements) per load, logical chunks CPL sc ...;
  // load i holds row RPL i + sr, whose swizzle key repeats every 16 / RPL loads for K
  // (row & 15) and every 8 / RPL (at least 1) loads for V (row & 7).
  constexpr int CPL = BFP8 ? 2 : 1;
  // swizzle keys of a tile row (period 16 rows for K, 8 for V)
  auto kkey = [](int row) { return D == 64 ? (row >> 1) & 7 : row & 15; };
  auto vkey = [](int row) {
    const int y = D == 64 ? (row >> 1) & 3 : row & 7;
    return (2 * y) | (y & 1);
  };
  constexpr int KPAT = RPL >= 16 ? 1 : 16 / RPL, VPAT = RPL >= 8 ? 1 : 8 / RPL;
  uint32_t kw[KPAT], vw[VPAT];
#pragma unroll
  for (int j = 0; j < KPAT; ++j)
    kw[j] = (uint32_t)(sr * ROWB + (((CPL * sc) ^ kkey(RPL * j + sr)) << 4));
#pragma unroll
  for (int j = 0; j < VPAT; ++j)
    vw[j] = (uint32_t)(sr * ROWB + (((CPL * sc) ^ vkey(RPL * j + sr)) << 4));
  // A-operand reads of K: row 16 b + n, chunk 4 s + quad
  uint32_t kr[KSTEPS];
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) kr[s] = (uint32_t)(n * ROWB + (((4 * s + quad) ^ kkey(n)) << 4));
  // transposing reads of V: lane addresses row 4 quad + n / 4 (+ 16 per key block), the 8 bytes
  // at element 16 db + 4 (n & 3)
  uint32_t vr[DBLK];
  {
    const int vrow = 4 * quad + (n >> 2), xx = (n & 3) >> 1;  // key blocks start at multiples of 16
#pragma unroll
    for (int db = 0; db < DBLK; ++db)
      vr[db] = (uint32_t)(vrow * ROWB + (((2 * db + xx) ^ vkey(vrow)) << 4) + 8 * (n & 1));
  }

  auto locate = [&](int64_t xx) { return locate_unit<TILE>(a, s_pref, s_len, xx, seg_units); };
  // `bad`: bit i set where run i's block lies outside the table or the cache (it reads block 0)
  auto tile_offsets = [&](const Cursor &cu, int64_t (&eo)[NOFF], int64_t (&xo)[NOFF], uint32_t &bad) {
    bad = 0;
    bool base_bad = false;
    const int32_t *pt_row = page_table + (int64_t)cu.u * a.pt_rs;
    const int tok0 = cu.t * TILE;
    // a run never crosses a block (block_size is a multiple of the run length), so block and
    // row advance without a division; the table is read again only where the block changes
    int col = block_of(a, tok0), row = tok0 - col * a.bs;
    int64_t base = 0;
#pragma unroll
    for (int i = 0; i < NOFF; ++i) {
      if (i == 0 || row == 0) {
        int phys = (col < a.w) ? __builtin_amdgcn_readfirstlane(pt_row[col]) : -1;
        base_bad = (unsigned)phys >= (unsigned)a.nb;
        if (base_bad) phys = 0;
        base = ((int64_t)phys * a.hkv + cu.h) * slab;
      }
      if (base_bad) bad |= 1u << i;
      eo[i] = base + (int64_t)row * D * BPE;
      xo[i] = base + (int64_t)a.bs * D + (int64_t)row * GPR;
      row += RPL * LPO;
      if (row >= a.bs) row = 0, ++col;
    }
  };
  auto fetch = [&](const uint8_t *base, const int64_t (&eo)[NOFF], const int64_t (&xo)[NOFF],
                   u32x4 (&raw)[NL], uint32_t (&ex)[NL]) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const uint8_t *erow = base + eo[i / LPO] + (i % LPO) * (RPL * D * BPE);
      raw[i] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4 *>(erow + static_cast<uint64_t>(lane_bytes)));
      if constexpr (BFP8) {
        const uint8_t *xrow = base + xo[i / LPO] + (i % LPO) * (RPL * GPR);
        ex[i] = __builtin_nontemporal_load(
            reinterpret_cast<const uint32_t *>(xrow + static_cast<uint64_t>(lane_exp)));
      }
    }
  };
  // FUSED: the lane's part of the fresh K or V row of (user, head): the 16 bytes of its chunk
  // for a bfloat16 cache, the 16 bfloat16 elements of its group for block-float-8.
  constexpr int NF = BFP8 ? 2 : 1;
  struct Fresh {
    u32x4 part[NF];
  };
  auto fetch_fresh = [&](const uint16_t *src, const Cursor &cu) {
    const uint16_t *p = src + cu.u * a.new_us + cu.h * a.new_hs + (BFP8 ? 16 : 8) * sc;
    Fresh f;
#pragma unroll
    for (int j = 0; j < NF; ++j) f.part[j] = *reinterpret_cast<const u32x4 *>(p + 8 * j);
    return f;
  };
  // FUSED: puts the fresh row (quantised here for block-float-8) in place of row `r_star` of
  // the fetched tile (registers) and stores it into the cache row `row` of the slab at byte
  // offset `slab_base`.
  auto patch_and_store = [&](uint8_t *cache, u32x4 (&raw)[NL], uint32_t (&ex)[NL], const Fresh &fresh,
                             int r_star, int64_t elem_off, int64_t exp_off) {
    const int i_star = r_star / RPL;
    const bool mine = sr == r_star % RPL;
    u32x4 val = fresh.part[0];
    uint32_t e = 0;
    if constexpr (BFP8) {
      const u32x4 lo = fresh.part[0], hi = fresh.part[NF - 1];
      const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      uint32_t out[4];
      e = bfp8_encode16<D == 256>(w, out);
      val = u32x4{out[0], out[1], out[2], out[3]};
    }
#pragma unroll
    for (int i = 0; i < NL; ++i)
      if (i == i_star && mine) {
        raw[i] = val;
        if constexpr (BFP8) ex[i] = e << exp_shift;
      }
    if (mine) {
      *reinterpret_cast<u32x4 *>(cache + elem_off + 16 * sc) = val;
      if constexpr (BFP8) cache[exp_off + sc] = (uint8_t)e;
    }
  };
  // Cuts the lane's exponent bytes out of the fetched dwords (zero for rows past `nvalid` of a
  // partial tile, which stages them as zeros) and returns the largest of the tile.
  auto tile_exponent = [&](uint32_t (&ex)[NL], int nvalid, bool partial) {
    uint32_t e = 0;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      ex[i] = (ex[i] >> exp_shift) & 0xffu;
      if (partial && RPL * i + sr >= nvalid) ex[i] = 0;
      e = max(e, ex[i]);
    }
    return (int)wave_max_u32(e);
  };
  // registers -> LDS.  Block-float-8: expanded to half precision relative to the exponent
  // `eref`: the group scale 2^(e - eref) is the half with exponent field e - eref + 15; groups
  // more than 2^14 below the tile's largest (field <= 0) are written as zeros.  bfloat16:
  // copied; `clear` writes the rows past `nvalid` as zeros (unattended V rows must not carry
  // Inf / NaN into the product).
  auto stage = [&](bool is_v, const u32x4 (&raw)[NL], const uint32_t (&ex)[NL], int eref, int nvalid,
                   bool clear) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const uint32_t w0 = (is_v ? vw[i % VPAT] : kw[i % KPAT]) + (uint32_t)(i * RPL * ROWB);
      if constexpr (BFP8) {
        const uint32_t field = (uint32_t)max((int)ex[i] - (eref - 15), 0);
        const uint32_t sbits = field << 10;
        const halfx2 s2 = __builtin_bit_cast(halfx2, sbits | (sbits << 16));
        const halfx2 c2 = s2 * halfx2{(_Float16)-1152.f, (_Float16)-1152.f};
        uint32_t o[8];
        expand4_half(raw[i].x, s2, c2, o[0], o[1]);
        expand4_half(raw[i].y, s2, c2, o[2], o[3]);
        expand4_half(raw[i].z, s2, c2, o[4], o[5]);
        expand4_half(raw[i].w, s2, c2, o[6], o[7]);
        *reinterpret_cast<uint4 *>(tile + w0) = make_uint4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<uint4 *>(tile + (w0 ^ 16u)) = make_uint4(o[4], o[5], o[6], o[7]);
      } else {
        const bool keep = !clear || RPL * i + sr < nvalid;
        *reinterpret_cast<uint4 *>(tile + w0) =
            keep ? make_uint4(raw[i].x, raw[i].y, raw[i].z, raw[i].w) : make_uint4(0, 0, 0, 0);
      }
    }
  };
  // Q fragments: B operand, lane%16 = head of the group (zero beyond G): as they are for a
  // bfloat16 cache; half precision, scaled by 2^(127 - eq) with eq the largest exponent field of
  // the segment's Q, for block-float-8.  (Requesting the next segment's Q rows early, ahead of
  // the tile loads and inside the branch that detects the segment change, was measured slower:
  // the wait-count pass then drains the tile loads in the steady-state loop.)
  int eq = 0;
  auto load_q = [&](const Cursor &cu, u32x4 (&qf)[KSTEPS]) {
    const uint16_t *qp =
        a.q + cu.u * a.q_us + (int64_t)(cu.h * G + min(n, G - 1)) * a.q_hs + 8 * quad;
    const uint32_t qmask = n < G ? 0xffffffffu : 0u;  // no branch: a branch would wait for every load in flight
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      const uint4 t = *reinterpret_cast<const uint4 *>(qp + 32 * s);
      qf[s] = u32x4{t.x & qmask, t.y & qmask, t.z & qmask, t.w & qmask};
    }
    if constexpr (BFP8) {
      uint32_t em = 0;
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          em = max(em, max((qf[s][j] >> 7) & 0xffu, (qf[s][j] >> 23) & 0xffu));
      eq = (int)min(wave_max_u32(em), 253u);
      const float qs = __builtin_bit_cast(float, (uint32_t)(254 - eq) << 23);
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          qf[s][j] = pack_half2(bf16_lo(qf[s][j]) * qs, bf16_hi(qf[s][j]) * qs);
    }
  };

  if constexpr (DIRECT == 0) cur = locate_unit<TILE>(a, s_pref, s_len, x_lo, seg_units, &x);
  int64_t eo[NOFF], xo[NOFF];
  u32x4 kraw[NL], vraw[NL];
  uint32_t kex[NL], vex[NL];
  u32x4 qf[KSTEPS];
  Fresh kfresh = {}, vfresh = {};
  uint32_t bad_cur = 0;  // the current tile's runs that read block 0 in place of a block out of range
  const bool works = DIRECT == 0 || cur.tiles_left > 0;  // (a short segment leaves wavefronts without a tile)
  if (works) {
    tile_offsets(cur, eo, xo, bad_cur);
    fetch(a.k, eo, xo, kraw, kex);
    fetch(a.v, eo, xo, vraw, vex);
    if constexpr (FUSED) {
      kfresh = fetch_fresh(a.k_new, cur);
      vfresh = fetch_fresh(a.v_new, cur);
    }
    load_q(cur, qf);
  }
  if constexpr (DIRECT == 0) publish_segment_row(a, s_pref, total, n_eff, seg_units);

  floatx4 acc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  int ev_run = 0;  // reference exponent of the V accumulator

  auto process_tile = [&](auto has_next_tag) {
    constexpr bool has_next = decltype(has_next_tag)::value;
    const int nvalid = cur.len - cur.t * TILE;
    const bool partial = nvalid < TILE;
    const int nbelow = cur.lo - cur.t * TILE;  // sliding window: > 0 only in a segment's first tile
    const bool same_seg = DIRECT > 0 || (has_next && cur.tiles_left > 1);
    Cursor nxt = cur;

    // ---- K: registers -> LDS, then the next tile's K: global -> registers -------------------
    // FUSED: is this the tile that holds the token at cur_pos (the segment's last), and is that
    // position inside the table and its block inside the cache?  The row's place in the cache
    // comes from the tile's own offsets: a second look at the position and the page table would
    // be two round trips to memory in the middle of the tile, each waiting for every load in
    // flight, and the wavefronts that end a segment are the ones a launch ends up waiting for.
    bool fresh_ok = false;
    int64_t fresh_eo = 0, fresh_xo = 0;
    if constexpr (FUSED) {
      if (cur.tiles_left == 1 && nvalid > 0) {
        // a length below the table's capacity is the position + 1; at the capacity it may have
        // been cut short, and only then the position is read again
        const int64_t cap = (int64_t)a.w * a.bs;
        const bool exact = cur.len < cap || load_index(cur_pos, a.cur_i64, cur.u) == cur.len - 1;
        constexpr int RUN_ROWS = RPL * LPO;
        const int i_run = (nvalid - 1) / RUN_ROWS, rr = (nvalid - 1) % RUN_ROWS;
        if (exact && !((bad_cur >> i_run) & 1u)) {
          fresh_ok = true;
#pragma unroll
          for (int i = 0; i < NOFF; ++i)
            if (i == i_run) fresh_eo = eo[i] + (int64_t)rr * D * BPE, fresh_xo = xo[i] + (int64_t)rr * GPR;
        }
      }
      if (fresh_ok) patch_and_store(const_cast<uint8_t *>(a.k), kraw, kex, kfresh, nvalid - 1, fresh_eo, fresh_xo);
    }
    int eref_k = 0, eref_v = 0;
    if constexpr (BFP8) eref_k = tile_exponent(kex, nvalid, partial);
    stage(false, kraw, kex, eref_k, nvalid, false);
    if constexpr (has_next) {
      if (same_seg) {
        constexpr int kStep = DIRECT > 0 ? DIRECT : 1;
        nxt.t = cur.t + kStep;
        nxt.tiles_left = cur.tiles_left - kStep;
      } else {
        nxt = locate(x + 1);
      }
      tile_offsets(nxt, eo, xo, bad_cur);  // (of the next tile: this one's has been used above)
      fetch(a.k, eo, xo, kraw, kex);
    }

    // ---- S^T = K . Q^T ------------------------------------------------------------------------
    floatx4 st[KBLK];
#pragma unroll
    for (int b = 0; b < KBLK; ++b) {
      st[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        const uint4 kq = *reinterpret_cast<const uint4 *>(tile + kr[s] + b * (16 * ROWB));
        st[b] = mma16<BFP8>(u32x4{kq.x, kq.y, kq.z, kq.w}, qf[s], st[b]);
      }
    }
    // ---- online softmax: lane (head, quad) holds keys 16 b + 4 quad + r ------------------------
    if (partial || nbelow > 0) {
#pragma unroll
      for (int b = 0; b < KBLK; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = 16 * b + 4 * quad + r;
          if (key >= nvalid || key < nbelow) st[b][r] = -INFINITY;
        }
    }
    // the factors taken out of the K tile and out of Q come back in the scale
    const float scale = BFP8 ? __builtin_ldexpf(a.scale_log2e, eref_k + eq - 260) : a.scale_log2e;
    if constexpr (MASKED) {  // the mask, brought to the units of the raw scores
      const float unit = 1.4426950408889634f / scale;
      const uint16_t *mrow = a.mask + cur.u * a.mask_us + (int64_t)(cur.h * G + min(n, G - 1)) * a.mask_hs +
                             cur.t * TILE + 4 * quad;
#pragma unroll
      for (int b = 0; b < KBLK; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * b + 4 * quad + r < nvalid) st[b][r] += bf16_lo(mrow[16 * b + r]) * unit;
    }
    float mloc = -INFINITY;
    if (scale >= 0.f) {
#pragma unroll
      for (int b = 0; b < KBLK; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, st[b][r]);
      mloc *= scale;
    } else {  // a negative scale turns the maximum into a minimum: compare scaled scores
#pragma unroll
      for (int b = 0; b < KBLK; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, st[b][r] * scale);
    }
    mloc = max_over_quads(mloc);
    const float m_new = fmaxf(m_run, mloc);
    const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_safe);
    m_run = m_new;

    // ---- V: registers -> LDS (the K tile has been consumed), next tile's V -> registers -------
    if constexpr (FUSED) {
      if (fresh_ok) patch_and_store(const_cast<uint8_t *>(a.v), vraw, vex, vfresh, nvalid - 1, fresh_eo, fresh_xo);
    }
    if constexpr (BFP8) eref_v = tile_exponent(vex, nvalid, partial);
    stage(true, vraw, vex, eref_v, nvalid, partial);
    if constexpr (has_next) fetch(a.v, eo, xo, vraw, vex);

    float lsum = 0.f, alpha_acc = alpha;
    u32x4 pf[PSTEPS];
    if constexpr (BFP8) {
      // bring this tile's V factor and the accumulator to the larger reference exponent
      const int ev_new = max(ev_run, eref_v);
      const float pscale = __builtin_ldexpf(1.f, eref_v - ev_new);
      alpha_acc = alpha * __builtin_ldexpf(1.f, ev_run - ev_new);
      ev_run = ev_new;
#pragma unroll
      for (int b = 0; b < KBLK; ++b)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(st[b][r], scale, -m_safe));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(st[b][r + 1], scale, -m_safe));
          lsum += p0 + p1;  // half-precision rounding of the weights is 2^-12: not tracked
          pf[b >> 1][2 * (b & 1) + (r >> 1)] = pack_half2(p0 * pscale, p1 * pscale);
        }
    } else {
#pragma unroll
      for (int b = 0; b < KBLK; ++b)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(st[b][r], scale, -m_safe));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(st[b][r + 1], scale, -m_safe));
          uint32_t w = pack_bf16x2(p0, p1);
          if constexpr (ONE) w = less_units(w, 0x00010001u);
          lsum += bf16_lo(w) + bf16_hi(w);  // the normaliser sums the weights that multiply V
          pf[b >> 1][2 * (b & 1) + (r >> 1)] = w;
          if constexpr (ONE) st[b][r] = p0 - bf16_lo(w), st[b][r + 1] = p1 - bf16_hi(w);  // the second parts
        }
    }
    l_run = l_run * alpha + lsum;
    if (__builtin_amdgcn_ballot_w64(alpha_acc != 1.0f) != 0) {
#pragma unroll
      for (int i = 0; i < DBLK; ++i) acc[i] *= alpha_acc;
    }
    // ---- O^T += V^T . P^T ------------------------------------------------------------------------
    auto second_product = [&]() {
#pragma unroll
      for (int s = 0; s < PSTEPS; ++s)
#pragma unroll
        for (int db = 0; db < DBLK; ++db) {
          typedef __attribute__((address_space(3))) shortx4 *lds_v4;
          const uint8_t *vp = tile + vr[db] + s * (32 * ROWB);
          shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(vp));
          shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(vp + 16 * ROWB));
          const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
          acc[db] = mma16<BFP8>(u32x4{l2.x, l2.y, h2.x, h2.y}, pf[s], acc[db]);
        }
    };
    second_product();
    // One query head per KV head (ONE): the weights in two bfloat16 parts.  The dot-product kernel, which serves such groups where this
    // one is not built, keeps a running maximum per sixteen of a tile's tokens, so more of its weights are exact; rounded once, this
    // kernel's results were 4 - 7 % further from a 64-bit evaluation than that one's (2.09e-3 against 1.97e-3, 128 tokens of 8 / 8
    // heads), in two parts they are 15 - 17 % closer (1.66e-3).  The first part is the rounded weight less one unit of its last
    // place, so that the second is positive: with zero or less, an infinite V element would come out as NaN.  A kernel of its own: as a
    // run-time branch the second parts cost every group 1 - 3 % (branch / kernels: 5 users of 32/8 heads in a window of 4096 19.1 / 18.9 us,
    // 8 of 64/8 of 64 with 512 ... 4096 17.0 / 16.7, 37 of 8/8 of 64 in a window of 512 14.5 / 14.0).
    if constexpr (ONE) {
      float low = 0.f;
#pragma unroll
      for (int b = 0; b < KBLK; ++b)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          low += st[b][r] + st[b][r + 1];
          pf[b >> 1][2 * (b & 1) + (r >> 1)] = pack_bf16x2(st[b][r], st[b][r + 1]);
        }
      l_run += low;
      second_product();
    }

    // ---- close the segment --------------------------------------------------------------------
    if (!same_seg) {
      float *slot = a.ws_slots + ((int64_t)wave + (int64_t)cur.u * a.hkv + cur.h) * a.slot_floats;
      const float l_tot = sum_over_quads(l_run);
      const float vout = BFP8 ? __builtin_ldexpf(1.f, ev_run - 133) : 1.f;
      if (n < G) {
        float *dst = slot + n * D + 4 * quad;
#pragma unroll
        for (int db = 0; db < DBLK; ++db)
          *reinterpret_cast<float4 *>(dst + 16 * db) = make_float4(
              acc[db][0] * vout, acc[db][1] * vout, acc[db][2] * vout, acc[db][3] * vout);
        if (quad == 0) {
          slot[G * D + n] = m_run;
          slot[G * D + G + n] = l_tot;
        }
      }
#pragma unroll
      for (int i = 0; i < DBLK; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
      m_run = -INFINITY;
      l_run = 0.f;
      ev_run = 0;
      if constexpr (has_next) {
        load_q(nxt, qf);
        if constexpr (FUSED) {  // the fresh rows of the new segment, once per segment
          kfresh = fetch_fresh(a.k_new, nxt);
          vfresh = fetch_fresh(a.v_new, nxt);
        }
      }
    }
    cur = nxt;
    x += same_seg ? 1 : 1 + seg_units;
  };
  if constexpr (DIRECT > 0) {
    if (works) {
      while (cur.tiles_left > DIRECT) process_tile(std::true_type{});
      process_tile(std::false_type{});
    }
    merge_waves<D, DIRECT>(a, cur.u, cur.h, G, std::min(n_tiles, DIRECT), tile, tiles, kTileBytes, acc,
                           BFP8 ? __builtin_ldexpf(1.f, ev_run - 133) : 1.f, m_run, sum_over_quads(l_run));
    return;
  }
  // the unit of the tile behind the current one: the next, or behind the next segment's leading units
  auto next_tile_unit = [&]() { return x + (cur.tiles_left > 1 ? 1 : 1 + seg_units); };
  while (next_tile_unit() < x_hi) process_tile(std::true_type{});
  process_tile(std::false_type{});
}

template <int D, bool BFP8, int RUNS, bool FUSED, bool MASKED = false, int DIRECT = 0, bool LONG = false, bool ONE = false>
bool launch(const DecodeArgs &a, hipStream_t st) {
  constexpr int kWaves = DIRECT ? DIRECT : kWavesPerBlock;
  const int blocks = DIRECT ? a.users * a.hkv : a.n_waves / kWavesPerBlock;
  const size_t lds = (size_t)kWaves * tile_bytes<D, LONG>();
  static std::atomic<uint64_t> lds_ready{0};
  const auto kernel = &paged_decode_mfma16_kernel<D, BFP8, RUNS, FUSED, MASKED, DIRECT, LONG, ONE>;
  if (!ensure_dynamic_lds(reinterpret_cast<const void *>(kernel), lds, lds_ready)) return false;
  launch_dominant(kernel, dim3(blocks), dim3(kWave * kWaves), lds, st, a, a.pt, a.cur);
  return true;
}

// Equal ranges of the flat list, or one workgroup per segment (DIRECT); the variant for the block size.
template <int D, bool BFP8, bool FUSED, int DIRECT, bool LONG, bool ONE>
bool launch_runs(const DecodeArgs &a, hipStream_t st) {
  constexpr int TILE = tile_bytes<D, LONG>() / (2 * D);
  if (a.bs % TILE == 0) return launch<D, BFP8, 1, FUSED, false, DIRECT, LONG, ONE>(a, st);
  if (DIRECT > 0 || a.bs % (TILE / 2) == 0) return launch<D, BFP8, 2, FUSED, false, DIRECT, LONG, ONE>(a, st);
  if constexpr (DIRECT == 0) {
    if (LONG || a.bs % (TILE / 4) == 0) return launch<D, BFP8, 4, FUSED, false, 0, LONG, ONE>(a, st);  // (block-float-8: blocks of 16 tokens)
    if constexpr (!LONG) return launch<D, BFP8, 0, FUSED, false, 0, false, ONE>(a, st);
  }
  return false;
}

// FUSED (a.k_new set): the launch also performs the cache update of the step.
template <int D, bool BFP8, bool FUSED>
bool launch_form(const DecodeArgs &a, hipStream_t st) {
  constexpr bool kOneHead = !BFP8;  // one query head per KV head has kernels of its own
  const bool one = kOneHead && a.hq == a.hkv;
  if (a.direct == 4) return one ? launch_runs<D, BFP8, FUSED, 4, false, kOneHead>(a, st) : launch_runs<D, BFP8, FUSED, 4, false, false>(a, st);
  if constexpr (D <= 128) {
    if (a.direct == 8) return one ? launch_runs<D, BFP8, FUSED, 8, false, kOneHead>(a, st) : launch_runs<D, BFP8, FUSED, 8, false, false>(a, st);
  }
  if constexpr (D == 128 && BFP8)
    if (a.long_tiles) return launch_runs<D, BFP8, FUSED, 0, true, false>(a, st);
  return one ? launch_runs<D, BFP8, FUSED, 0, false, kOneHead>(a, st) : launch_runs<D, BFP8, FUSED, 0, false, false>(a, st);
}

template <int D, bool BFP8>
bool launch_for_block_size(const DecodeArgs &a, hipStream_t st) {
  if (a.mask != nullptr) return a.k_new == nullptr && launch<D, BFP8, 0, false, true>(a, st);
  return a.k_new ? launch_form<D, BFP8, true>(a, st) : launch_form<D, BFP8, false>(a, st);
}

}  // namespace
}  // namespace decode
}  // namespace ttpa
