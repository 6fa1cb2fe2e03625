// The decode step of a latent layer in one call: around the latent attention kernels (decode_wide.hip)
// the projections of the layer, without the concatenated copies in between.
//
//   latent_query_kernel  q_lat[u, n] = (q_nope[u, n] . W_UK[n], q_rope[u, n]), and the new token's row
//                        (latent, rope) of every user goes into the paged cache
//   latent attention     o_lat[u, n] over the paged cache (its own launches)
//   latent_value_kernel  out[u, n] = o_lat[u, n] . W_UV[n]
//
// Both kernels are short: 2 MB of weights and 2 - 4 MB of activations for 128 users of 16 heads, bounded by
// the trip to memory and back.  So the split is for many small workgroups: (128 latent columns, head, 32
// users) for the query, (32 value columns, head, 32 users) with the contraction over the latent width cut
// between the four wavefronts for the value.  A weight tile travels memory -> LDS directly and is read
// through the transposing LDS load, so that v_mfma_f32_32x32x16_bf16 gets the users as its columns and
// the activations go from memory to registers as they are.
// A weight whose contracted dimension is the contiguous one (how a joint projection [heads * (128 + 128), 512] leaves W_UV
// after a split and a transposition, and [512, heads, 128 + 128] leaves W_UK) is the operand that the matrix instruction
// wants: lane (column, half) takes 8 consecutive elements per step, from memory to registers, without LDS.  (A copy into
// the other layout took a pass over the weights, 2 MB at 16 heads and 16 MB at 128, in front of every step: captured steps
// with either of these layouts, one user over 512 tokens at 16 heads 33.8 -> 27.1 us, 128 users 86.4 -> 79.4, one user at 128
// heads 83.2 -> 52.0 and 81.1 -> 48.4; with rows contiguous 26.7, 78.8 and 49.9.)  128 users, 16 heads: 8.2 and 5.0 us, where two
// batched library products, two concatenations, the cache write and the copy to the output took 41 us in six
// launches; the whole pass over contexts of 512 .. 8192 168 -> 94 us, of one user over 512 tokens 149 -> 37 us.
//
// And the prompt pass of a latent layer in one call.  Up to 64 tokens in the absorbed form (two kernels of the step around
// ttpa_latent_prefill, with the tokens as users), longer ones with K and V expanded per head:
//
//   latent_expand_kernel  k[t, n] = latent[t] . W_UK[n], v[t, n] = latent[t] . W_UV[n], and the prompt's rows go into the cache
//   ttpa_split_key_prefill over (k, rope) and v
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace ttpa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

constexpr int kNope = 128, kRope = 64, kLatent = 512, kValue = 128;
constexpr int kRow = kLatent + kRope;
constexpr int kUsers = 32;  // users per workgroup: the 32-wide dimension of the matrix instruction

struct StepArgs {
  const uint16_t *q_nope, *q_rope, *latent, *rope, *w_uk, *w_uv;
  int64_t qn_us, qn_hs, qr_us, qr_hs, latent_us, rope_us;
  int64_t uk_hs, uk_ld, uv_hs, uv_ld;  // head stride, and the stride of the dimension that is not contiguous
  uint16_t *q_lat, *o_lat;  // [users][heads][kRow], [users][heads][kLatent]
  uint16_t *out;
  int64_t out_us, out_hs;
  uint16_t *cache;
  const int32_t *pt;
  int64_t pt_rs;
  const void *pos;
  int pos_i64;
  int users, heads, bs, w, nb;
  int tiles;  // blocks of 32 users per workgroup of latent_value_kernel
  // prompt: the rows are tokens, `seq` to a user, and belong to positions 0 .. seq - 1 of the users' table rows
  int seq, table_rows;
  uint16_t *k_lat;  // [rows][kRow]
};

// Block and row of the cache for row v of a prompt pass (the fill's rule); false: outside the table or the cache.
__device__ __forceinline__ bool prompt_slot(const StepArgs &a, int v, int &phys, int &row) {
  const int u = v / a.seq, t = v - u * a.seq, col = t / a.bs;
  if (!a.cache || u >= a.table_rows) return false;
  phys = a.pt[u * a.pt_rs + col], row = t - col * a.bs;
  return (unsigned)phys < (unsigned)a.nb;
}

// A operand of a 32x32x16 instruction from rows 16 s .. 16 s + 15 (k) and 32 columns (m) of a weight tile in LDS:
// lane (m, h) receives column m of rows 8 h .. 8 h + 7.  `first` addresses the lane's 8 bytes of rows
// 8 h .. 8 h + 3 (row 8 h + (lane % 16) / 4), `half` is the byte distance of four rows.
__device__ __forceinline__ bf16x8 read_transposed(const unsigned char *first, int half) {
  typedef __attribute__((address_space(3))) shortx4 *lds_v4;
  const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)first);
  const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(first + half));
  struct {
    shortx4 a, b;
  } t = {lo, hi};
  return __builtin_bit_cast(bf16x8, t);
}

// The eight A operands of a wavefront where the contracted dimension is contiguous: `column` is the lane's column (32 of
// them `ld` elements apart), at the lane's first element of the contracted dimension.
__device__ __forceinline__ void load_columns(bf16x8 (&w)[8], const uint16_t *column) {
#pragma unroll
  for (int s = 0; s < 8; ++s) w[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(column + 16 * s));
}

// Activation rows travel memory -> LDS in whole rows of 256 bytes, four to an instruction, and results leave as whole rows: as 16 bytes of each of
// 32 rows per instruction (8 bytes for the results), each wavefront for itself, they were half of the query's time (128 heads,
// 75 users 14.9 -> 10.8 us; 16 heads, 128 users 7.6 -> 6.8; a prompt of 32 tokens of 16 heads 24.2 -> 22.8 for the whole pass).
// 16-byte chunk c of row r lies at chunk position c ^ (r % 16): the lanes of a fragment read find their rows in different banks.
constexpr int kRowPitch = 272;  // of result rows: 8-byte writes of 32 rows spread over the banks

// Pieces first ... first + count - 1 (four rows each) of the 32 rows of 128 elements from user u0 on, `us` elements apart.  Users past the
// last repeat it in the last piece, and nothing is read for further ones: a column of the products is a user's, and theirs are not stored.
__device__ __forceinline__ void request_rows(const uint16_t *src, int64_t us, int u0, int users, unsigned char *rows, int first, int count) {
  const int lane = threadIdx.x & 63;
  for (int j = first; j < min(first + count, (users - u0 + 3) >> 2); ++j) {
    const int r = 4 * j + (lane >> 4);
    dma16_lane(src + min(u0 + r, users - 1) * us + 8 * ((lane & 15) ^ (r & 15)),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_address(rows) + 1024u * (uint32_t)j)));
  }
}
__device__ __forceinline__ bf16x8 read_row(const unsigned char *rows, int r, int chunk) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(rows + r * 256 + 16 * (chunk ^ (r & 15))));
}

// COLUMNS: the weight's contracted dimension is contiguous (else its columns are).  PROMPT: the rows' latent keys go to a.k_lat
// as well, in one piece for the attention.
template <bool COLUMNS, bool PROMPT = false>
__global__ __launch_bounds__(256) void latent_query_kernel(StepArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char tile[COLUMNS ? 1024 : kNope * 256];  // 128 rows of 128 columns
  __shared__ __attribute__((aligned(1024))) unsigned char rows[kUsers * kRowPitch];            // the users' query rows, then their result rows
  const int col0 = blockIdx.x * 128, head = blockIdx.y, u0 = blockIdx.z * kUsers;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;

  // weights: 32 segments of four rows; 16-byte chunk c of row r lies at chunk position c ^ 4 (r % 4), which puts the
  // four rows of a transposing read in different banks
  bf16x8 columns[8];
  if constexpr (COLUMNS) {
    load_columns(columns, a.w_uk + head * a.uk_hs + (int64_t)(col0 + 32 * wave + n) * a.uk_ld + 8 * h);
  } else {
    const uint16_t *w = a.w_uk + head * a.uk_hs + col0;
    const uint32_t lane_bytes = (uint32_t)(lane >> 4) * (uint32_t)(2 * a.uk_ld) + 16u * (uint32_t)((lane & 15) ^ (4 * (lane >> 4)));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int seg = 8 * wave + j;
      dma16_uniform(w + (int64_t)(4 * seg) * a.uk_ld, lane_bytes, lds_address(tile) + 1024u * (uint32_t)seg);
    }
  }
  request_rows(a.q_nope + head * a.qn_hs, a.qn_us, u0, a.users, rows, 2 * wave, 2);

  if (blockIdx.x == 0) {  // the rotary part of the query, as it is: 8 chunks per user
    const int v = u0 + (tid >> 3), c = 8 * (tid & 7);
    if (v < a.users)
      *reinterpret_cast<uint4 *>(a.q_lat + ((int64_t)v * a.heads + head) * kRow + kLatent + c) =
          *reinterpret_cast<const uint4 *>(a.q_rope + v * a.qr_us + head * a.qr_hs + c);
  }
  // The new token's row: 128 latent columns per workgroup, the rotary part with the first.  (Parked users that share a
  // slot of the null block write it in any order.)
  if (head == 0) {
    const int chunks = 16 + (blockIdx.x == 0 ? 8 : 0);
    for (int i = tid; i < kUsers * chunks; i += 256) {
      const int v = u0 + i / chunks, c = i % chunks;
      int phys, row;
      if (v >= a.users) continue;
      if (!PROMPT && !update_slot(a.pos, a.pos_i64, a.pt, a.pt_rs, a.bs, a.w, a.nb, v, phys, row)) continue;
      const int at = c < 16 ? col0 + 8 * c : kLatent + 8 * (c - 16);
      const uint16_t *src = c < 16 ? a.latent + v * a.latent_us + at : a.rope + v * a.rope_us + 8 * (c - 16);
      const uint4 piece = *reinterpret_cast<const uint4 *>(src);
      if constexpr (PROMPT) {
        *reinterpret_cast<uint4 *>(a.k_lat + (int64_t)v * kRow + at) = piece;
        if (!prompt_slot(a, v, phys, row)) continue;
      }
      *reinterpret_cast<uint4 *>(a.cache + ((int64_t)phys * a.bs + row) * kRow + at) = piece;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's rows and segments have landed
  __syncthreads();
  bf16x8 q[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) q[s] = read_row(rows, n, 2 * s + h);

  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const int grp = lane >> 4, a16 = lane & 15;
  const int row = 8 * (grp >> 1) + (a16 >> 2), chunk = 4 * wave + 2 * (grp & 1) + ((a16 & 3) >> 1);
  const unsigned char *first = tile + row * 256 + 16 * (chunk ^ (4 * (row & 3))) + 8 * (a16 & 1);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    bf16x8 w;
    if constexpr (COLUMNS) w = columns[s];
    else w = read_transposed(first + s * 16 * 256, 4 * 256);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, q[s], acc, 0, 0, 0);
  }
  __syncthreads();  // everybody has its query rows
#pragma unroll
  for (int j = 0; j < 4; ++j)
    *reinterpret_cast<uint2 *>(rows + n * kRowPitch + 64 * wave + 16 * j + 8 * h) =
        make_uint2(pack_bf16x2(acc[4 * j], acc[4 * j + 1]), pack_bf16x2(acc[4 * j + 2], acc[4 * j + 3]));
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kUsers / 16; ++i) {
    const int v = 16 * i + (tid >> 4), c = tid & 15;
    if (u0 + v < a.users)
      *reinterpret_cast<uint4 *>(a.q_lat + ((int64_t)(u0 + v) * a.heads + head) * kRow + col0 + 8 * c) =
          *reinterpret_cast<const uint4 *>(rows + v * kRowPitch + 16 * c);
  }
}

// A workgroup takes a.tiles blocks of 32 users: the weight goes to registers once, and the rows of the next block are on their way while
// one is worked on.  128 heads, 75 users: 21.0 us with one block per workgroup (the weights read once per 32 users, three rounds of
// workgroups), 12.9.  (The query's kernel, which writes more than it reads, lost by the same: 10.8 / 16.2 us.)
template <bool COLUMNS>
__global__ __launch_bounds__(256) void latent_value_kernel(StepArgs a) {
  constexpr int kPitch = 36;  // floats of a user's partial sums: rows of 16-byte writes in different banks
  // Per wavefront 128 latent values of the users, then its partial sums, in two buffers in turn; the second holds the weight at first (512 rows
  // of 32 columns, 128 per wavefront), until it is in registers.
  __shared__ __attribute__((aligned(1024))) unsigned char buffer[2][4][kUsers * 256];
  static_assert(kUsers * kPitch * 4 <= kUsers * 256, "a wavefront's sums take its rows' place");
  const int col0 = blockIdx.x * 32, head = blockIdx.y, first_user = blockIdx.z * a.tiles * kUsers;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  // weights: 8 segments of sixteen 64-byte rows per wavefront (four rows of a transposing read are 256 consecutive bytes)
  bf16x8 w[8];
  if constexpr (COLUMNS) {
    load_columns(w, a.w_uv + head * a.uv_hs + (int64_t)(col0 + n) * a.uv_ld + 128 * wave + 8 * h);
  } else {
    const uint16_t *weight = a.w_uv + head * a.uv_hs + (int64_t)(128 * wave) * a.uv_ld + col0;
    const uint32_t lane_bytes = (uint32_t)(lane >> 2) * (uint32_t)(2 * a.uv_ld) + 16u * (uint32_t)(lane & 3);
#pragma unroll
    for (int j = 0; j < 8; ++j) dma16_uniform(weight + (int64_t)(16 * j) * a.uv_ld, lane_bytes, lds_address(buffer[1][wave]) + 1024u * j);
  }
  auto request = [&](int t) {
    request_rows(a.o_lat + (int64_t)head * kLatent + 128 * wave, (int64_t)a.heads * kLatent, first_user + t * kUsers, a.users, buffer[t & 1][wave], 0, 8);
  };
  request(0);
  const int tiles = min(a.tiles, (a.users - first_user + kUsers - 1) / kUsers);
  for (int t = 0; t < tiles; ++t) {
    const int u0 = first_user + t * kUsers;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // a wavefront reads the rows and segments that it requested
    if (!COLUMNS && t == 0) {
      const int grp = lane >> 4, a16 = lane & 15;
      const unsigned char *first = buffer[1][wave] + (8 * (grp >> 1) + (a16 >> 2)) * 64 + 32 * (grp & 1) + 8 * (a16 & 3);
#pragma unroll
      for (int s = 0; s < 8; ++s) w[s] = read_transposed(first + s * 16 * 64, 4 * 64);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if (t + 1 < tiles) request(t + 1);  // (its buffer: the weight is in registers, the sums of block t - 1 were read in front of a barrier)
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[s], read_row(buffer[t & 1][wave], n, 2 * s + h), acc, 0, 0, 0);
    auto sums = [&](int k) { return reinterpret_cast<float *>(buffer[t & 1][k]); };
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<float4 *>(sums(wave) + n * kPitch + 8 * j + 4 * h) = make_float4(acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]);
    __syncthreads();
    const int v = tid >> 3, c = 4 * (tid & 7);
    float4 x = *reinterpret_cast<const float4 *>(sums(0) + v * kPitch + c);
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      const float4 y = *reinterpret_cast<const float4 *>(sums(k) + v * kPitch + c);
      x.x += y.x, x.y += y.y, x.z += y.z, x.w += y.w;
    }
    if (u0 + v < a.users)
      *reinterpret_cast<uint2 *>(a.out + (u0 + v) * a.out_us + head * a.out_hs + col0 + c) = make_uint2(pack_bf16x2(x.x, x.y), pack_bf16x2(x.z, x.w));
    if (t + 1 < tiles) __syncthreads();
  }
}

// K and V of a prompt, expanded per head, and the fill of the cache in the same launch (34 GFLOP at 8192 tokens of 16 heads, 75 MB
// moved: 52 us, where two library products, a copy of W_UV, the fill and the gaps between them took 61).  Bound by the way of the
// operands from L2 into LDS, about 44 bytes per ns and CU: without its products the launch takes 45 us.  A workgroup
// computes 128 tokens x the 128 features of K or of V of a head, in steps of 32 or 64 latent values (ExpandShape); both operands travel
// memory -> LDS directly, in a ring of four or two steps, one barrier per step; 64 KiB, so two workgroups share a CU.  A
// slice's (16 values) fragments are read while the products of the slice before run.  A wavefront takes 64 x 64 as 2 x 2
// v_mfma_f32_32x32x16_bf16 tiles, features as rows, tokens as columns; the results meet in LDS so that stores are whole rows (57 us
// with 16 bytes per row and store).  Workgroups are ordered weights first: with the round-robin deal an XCD's L2 holds an
// eighth of the weights, and the tokens pass through it.  Not better: 256 tokens x K and V per workgroup, with half the bytes
// (49 us, but one workgroup per CU: 20 against 14 us for a pass of 96 tokens), and two workgroups per CU that go
// through their items without emptying the ring (56 us).
struct ExpandArgs {
  StepArgs s;                // latent, rope, weights, cache, table, rows (users), seq
  uint16_t *k, *v;           // [rows][heads][128]
  int uk_rows, uv_rows;      // the weight's contracted dimension is contiguous (else its features are)
  int items;                 // workgroups behind them write rows of the cache, 8 threads to a row
};

// Steps of 64 latent values in a ring of two where workgroups share CUs, in most of one round of the chip's 512 places or in two with the second more than
// half full: whole 128-byte lines per request instead of halves, which is worth more there than three steps on their way; a workgroup with a CU to itself, all
// of them up to 256 and the last ones of a launch that is a little over a round (the cache rows' workgroups come on top), depends on what it has on its
// way.  us per pass, steps of 32 / 64 (workgroups), / on another card: 16 heads, 1 x 1152 tokens 36.8 / 36.1, 37.7 / 36.1 (288), 4 x 320 24.1 / 23.4, 24.7 / 23.8 (320),
// 1 x 1536 43.9 / 43.4 (384), 4 x 448 27.2 / 26.2 (448); 2 x 1568 62.9 / 61.1 (800), 2 x 1760 71.1 / 69.6 (896), 2 x 2048 88.3 / 86.6 (1024), 3 x 1824 107.7 / 105.1 (1376),
// 4 x 2048 150.5 / 148.9, 145.0 / 149.3 (2048), 32 heads, 3 x 832 69.1 / 67.1 (1280), 128 heads, 1 x 416 46.6 / 44.7 (1024).  Neither: 16 heads, 1 x 96 12.5 / 12.9 (32),
// 1 x 512 21.3 / 22.3 (128), 1 x 896 28.9 / 29.9 (224); 1 x 1920 51.6 / 51.6, 50.6 / 49.8 (480), 2 x 1024 38.6 / 40.6,
// 36.2 / 36.1 (512), 2 x 1088 45.0 / 46.6, 43.3 / 43.1 (544), 1 x 2432 70.9 / 74.5, 67.4 / 67.6 (608), 2 x 1440 58.3 / 58.4 (720), 32 heads, 4 x 256 27.0 / 28.3, 25.4 / 25.4
// (512), 128 heads, 1 x 352 37.5 / 38.2 (768).  256 tokens per workgroup with steps of 32 or 64: 4 x 2048 the kernel alone 43.3 and 48.2 us against 45.4 and 41.7
// (the two above), 1 x 480 9.7 and 10.3 against 6.2 and 8.1.
constexpr int kExpTokens = 128;
template <int STEP, int STAGES>
struct ExpandShape {
  static constexpr int kStep = STEP, kStages = STAGES, kSteps = kLatent / STEP;
  static constexpr int kHalf = kExpTokens * STEP * 2, kStage = 2 * kHalf;  // bytes of the tokens' and of the weight's part of a step
  static constexpr int kPitch = 272;  // bytes of a result row in LDS: 8-byte writes of 32 rows spread over the banks
  static constexpr int kLds = kStages * kStage;
  static constexpr int kPieces = kHalf / 1024 / 2;  // requests of a wavefront per step
  static_assert(kExpTokens * kPitch <= kLds, "the results take the ring's place");
};

// Rows of 2 STEP bytes: 16-byte chunk c of row r lies at chunk position c ^ (r / 4 % 4) (64 bytes) or c ^ (r / 2 % 8) (128), so the lanes that
// LDS serves together find their chunks in different banks.
template <int STEP>
__device__ __forceinline__ int row_swizzle(int row) { return STEP == 32 ? (row >> 2) & 3 : (row >> 1) & 7; }
template <int STEP>
__device__ __forceinline__ bf16x8 read_row_chunk(const unsigned char *tile, int row, int chunk) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(tile + row * (2 * STEP) + 16 * (chunk ^ row_swizzle<STEP>(row))));
}

// part: 0 for K, 1 for V; ROWS: its weight's contracted dimension is contiguous.
template <class S, bool ROWS>
__device__ __forceinline__ void expand_item(const ExpandArgs &a, unsigned char *ring, int head, int part, int row0) {
  const StepArgs &p = a.s;
  constexpr int STEP = S::kStep;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Requests: the first two wavefronts bring the tokens' part of a step, the others the weight's.  A piece is 1 KiB, whole rows of 2 STEP bytes
  // or (a weight whose features are contiguous) four rows of 256.
  const bool weights = wave >= 2, by_row = !weights || ROWS;
  const int first = S::kPieces * (wave & 1);
  const int64_t ld = part ? p.uv_ld : p.uk_ld;
  const uint16_t *weight = part ? p.w_uv + head * p.uv_hs : p.w_uk + head * p.uk_hs;
  const uint64_t at = reinterpret_cast<uint64_t>(weights ? weight : p.latent + row0 * p.latent_us);
  const unsigned char *base = reinterpret_cast<const unsigned char *>(
      address_from_words(__builtin_amdgcn_readfirstlane((int)(uint32_t)at), __builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32))));
  const int64_t step_bytes = by_row ? 2 * STEP : 2 * ld * STEP;
  uint32_t lane_bytes[S::kPieces];
  {
    constexpr int kLanes = STEP / 8, kRows = 64 / kLanes;  // lanes per row, rows per piece
    const uint32_t pitch = (uint32_t)(weights ? 2 * ld : 2 * p.latent_us);
    const int last = weights ? kLatent : min(kExpTokens, p.users - row0) - 1;  // (rows behind the prompt repeat its last)
    const int per = by_row ? kRows : 4, in = by_row ? lane / kLanes : lane >> 4;
#pragma unroll
    for (int i = 0; i < S::kPieces; ++i) {
      const int r = per * (first + i) + in;
      const uint32_t chunk = by_row ? (lane % kLanes) ^ row_swizzle<STEP>(r) : (lane & 15) ^ (4 * (lane >> 4));
      lane_bytes[i] = (uint32_t)min(r, last) * pitch + 16u * chunk;
    }
  }
  const uint32_t to = lds_address(ring) + 1024u * (uint32_t)first + (weights ? (uint32_t)S::kHalf : 0u);
  auto request = [&](int step) {  // called for the steps in turn
    const uint32_t dst = to + (uint32_t)(step % S::kStages) * S::kStage;
#pragma unroll
    for (int i = 0; i < S::kPieces; i += 4) {
      const void *const bases[4] = {base, base - 1024, base - 2048, base - 3072};
      const uint32_t lanes[4] = {lane_bytes[i], lane_bytes[i + 1], lane_bytes[i + 2], lane_bytes[i + 3]};
      dma16_quad(bases, lanes, (uint32_t)__builtin_amdgcn_readfirstlane((int)(dst + 1024u * i)));
    }
    base += step_bytes;
  };

  const int n = lane & 31, h = lane >> 5, grp = lane >> 4, a16 = lane & 15;
  const int f0 = 64 * (wave & 1), t0 = 64 * (wave >> 1);  // the wavefront's features and tokens
  const int trow = 8 * (grp >> 1) + (a16 >> 2), tchunk = f0 / 8 + 2 * (grp & 1) + ((a16 & 3) >> 1);
  constexpr int kSlices = STEP / 16;  // products of a step
  floatx16 acc[2][2];
  bf16x8 w[2][2], x[2][2];  // the fragments of two slices in turn
  auto read = [&](int step, int slice) {
    const unsigned char *tokens = ring + step % S::kStages * S::kStage, *wtile = tokens + S::kHalf;
    const int to = slice & 1;
#pragma unroll
    for (int g = 0; g < 2; ++g) x[to][g] = read_row_chunk<STEP>(tokens, t0 + 32 * g + n, 2 * slice + h);
#pragma unroll
    for (int f = 0; f < 2; ++f)
      if constexpr (ROWS) w[to][f] = read_row_chunk<STEP>(wtile, f0 + 32 * f + n, 2 * slice + h);
      else w[to][f] = read_transposed(wtile + (16 * slice + trow) * 256 + 16 * ((tchunk + 4 * f) ^ (4 * (trow & 3))) + 8 * (a16 & 1), 4 * 256);
  };
  auto products = [&](int half) {
    __builtin_amdgcn_sched_barrier(0);  // (the scheduler would put the reads of the next slice behind these products)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int g = 0; g < 2; ++g) acc[f][g] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[half][f], x[half][g], acc[f][g], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // at most `steps` steps' requests of this wavefront are still under way, and its reads have returned
  auto wait = [&](auto steps) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(steps)::value * S::kPieces) : "memory");
  };
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[f][g][r] = 0.f;
#pragma unroll
  for (int step = 0; step < S::kStages; ++step) request(step);
  wait(std::integral_constant<int, S::kStages - 1>{});
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read(0, 0);
#pragma unroll
  for (int step = 0; step < S::kSteps; ++step) {
#pragma unroll
    for (int slice = 0; slice + 1 < kSlices; ++slice) {
      read(step, slice + 1);
      products(slice & 1);
    }
    if (step + 1 < S::kSteps) {
      // This wavefront's requests of the next step have landed and its reads of this one have returned; behind the
      // barrier that holds for everybody: the next step can be read, and this one's place filled.
      if (step + S::kStages - 1 < S::kSteps) wait(std::integral_constant<int, S::kStages - 2>{});
      else if (step + 2 < S::kSteps && S::kStages > 3) wait(std::integral_constant<int, 1>{});
      else wait(std::integral_constant<int, 0>{});
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (step + S::kStages < S::kSteps) request(step + S::kStages);
      read(step + 1, 0);
    }
    products((kSlices - 1) & 1);
  }
  // lane (n, h) holds features 8 j + 4 h ... + 3 of token n; the results meet in LDS so that stores are whole rows
  __syncthreads();
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<uint2 *>(ring + (t0 + 32 * g + n) * S::kPitch + 2 * (f0 + 32 * f + 8 * j + 4 * h)) =
            make_uint2(pack_bf16x2(acc[f][g][4 * j], acc[f][g][4 * j + 1]), pack_bf16x2(acc[f][g][4 * j + 2], acc[f][g][4 * j + 3]));
  __syncthreads();
  uint16_t *out = (part ? a.v : a.k) + head * 128 + 8 * (tid & 15);
#pragma unroll
  for (int i = 0; i < kExpTokens / 16; ++i) {
    const int r = (tid >> 4) + 16 * i;
    if (row0 + r < p.users)
      *reinterpret_cast<uint4 *>(out + (int64_t)(row0 + r) * p.heads * 128) = *reinterpret_cast<const uint4 *>(ring + r * S::kPitch + 16 * (tid & 15));
  }
}

template <class S>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void latent_expand_kernel(ExpandArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];
  const StepArgs &p = a.s;
  if ((int)blockIdx.x >= a.items) {
    const int tid = threadIdx.x, v = 32 * ((int)blockIdx.x - a.items) + (tid >> 3);
    int phys, row;
    if (v >= p.users || !prompt_slot(p, v, phys, row)) return;
    uint16_t *dst = p.cache + ((int64_t)phys * p.bs + row) * kRow + 8 * (tid & 7);
    const uint16_t *lat = p.latent + v * p.latent_us + 8 * (tid & 7);
    uintx4 piece[8];
    const uintx4 last = *reinterpret_cast<const uintx4 *>(p.rope + v * p.rope_us + 8 * (tid & 7));
#pragma unroll
    for (int c = 0; c < 8; ++c) piece[c] = *reinterpret_cast<const uintx4 *>(lat + 64 * c);
#pragma unroll
    for (int c = 0; c < 8; ++c) *reinterpret_cast<uintx4 *>(dst + 64 * c) = piece[c];
    *reinterpret_cast<uintx4 *>(dst + kLatent) = last;
    return;
  }
  const int wt = 2 * p.heads, which = (int)blockIdx.x % wt, row0 = (int)blockIdx.x / wt * kExpTokens;
  const int head = which >> 1, part = which & 1;
  if (part ? a.uv_rows : a.uk_rows) expand_item<S, true>(a, ring, head, part, row0);
  else expand_item<S, false>(a, ring, head, part, row0);
}

template <class S>
int launch_expand(ExpandArgs &e, hipStream_t st) {
  static std::atomic<uint64_t> lds_ready{0};
  if (!ensure_dynamic_lds(reinterpret_cast<const void *>(&latent_expand_kernel<S>), S::kLds, lds_ready))
    return fail(TTPA_ERR_LAUNCH, "latent prompt: cannot configure the expansion kernel");
  const int64_t groups = e.items + (e.s.cache ? ((int64_t)e.s.users + 31) / 32 : 0);
  latent_expand_kernel<S><<<dim3((unsigned)groups), dim3(256), S::kLds, st>>>(e);
  return check_launch("latent_prompt (expansion)");
}

// Blocks of 32 users per workgroup of latent_value_kernel, and how many workgroups share them: as many as keep two workgroups on every CU (their
// LDS), one where that leaves CUs idle.
inline unsigned lay_out_tiles(StepArgs &a) {
  const int64_t tiles = (a.users + kUsers - 1) / kUsers, wgs = 4 * (int64_t)a.heads * tiles;
  a.tiles = (int)std::min<int64_t>((wgs + 511) / 512, tiles);
  return (unsigned)((tiles + a.tiles - 1) / a.tiles);
}

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace
}  // namespace ttpa

using namespace ttpa;

extern "C" size_t ttpa_latent_decode_step_workspace_bytes(int32_t users, int32_t heads) {
  if (users <= 0 || heads <= 0) return 0;
  const size_t attn = ttpa_paged_mla_decode_workspace_bytes(users, heads, 1, kLatent);
  if (attn == 0) return 0;
  return align256(attn) + align256((size_t)users * heads * kRow * 2) + align256((size_t)users * heads * kLatent * 2);
}

#define TTPA_LATENT_STEP_HEAD                                                                                          \
  void *out, int64_t out_user_stride, int64_t out_head_stride, const void *q_nope, int64_t q_nope_user_stride,          \
      int64_t q_nope_head_stride, const void *q_rope, int64_t q_rope_user_stride, int64_t q_rope_head_stride,           \
      const void *latent, int64_t latent_user_stride, const void *rope, int64_t rope_user_stride, const void *w_uk
#define TTPA_LATENT_STEP_TAIL                                                                                          \
  void *cache, const int32_t *page_table, int64_t page_table_row_stride, const void *cur_pos, int cur_pos_is_i64,       \
      int32_t users, int32_t heads, int32_t block_size, int32_t table_width, int32_t num_blocks, float scale,           \
      void *workspace, size_t workspace_bytes, void *stream

extern "C" int ttpa_latent_decode_step(TTPA_LATENT_STEP_HEAD, int64_t w_uk_head_stride, int64_t w_uk_row_stride, const void *w_uv,
                                       int64_t w_uv_head_stride, int64_t w_uv_row_stride, TTPA_LATENT_STEP_TAIL) {
  return ttpa_latent_decode_step_strided(
      out, out_user_stride, out_head_stride, q_nope, q_nope_user_stride, q_nope_head_stride, q_rope, q_rope_user_stride,
      q_rope_head_stride, latent, latent_user_stride, rope, rope_user_stride, w_uk, w_uk_head_stride, w_uk_row_stride, 1, w_uv,
      w_uv_head_stride, w_uv_row_stride, 1, cache, page_table, page_table_row_stride, cur_pos, cur_pos_is_i64, users, heads,
      block_size, table_width, num_blocks, scale, workspace, workspace_bytes, stream);
}

extern "C" int ttpa_latent_decode_step_strided(TTPA_LATENT_STEP_HEAD, int64_t w_uk_head_stride, int64_t w_uk_row_stride,
                                               int64_t w_uk_column_stride, const void *w_uv, int64_t w_uv_head_stride,
                                               int64_t w_uv_row_stride, int64_t w_uv_column_stride, TTPA_LATENT_STEP_TAIL) {
  TTPA_REQUIRE(out && q_nope && q_rope && latent && rope && w_uk && w_uv && cache && page_table && cur_pos, "null pointer argument");
  TTPA_REQUIRE(users > 0 && heads > 0 && block_size > 0 && table_width > 0 && num_blocks > 0, "non-positive dimension");
  TTPA_REQUIRE(aligned16(q_nope) && aligned16(q_rope) && aligned16(latent) && aligned16(rope) && aligned16(w_uk) && aligned16(w_uv) &&
                   aligned16(cache) && (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
               "latent step: operands must be 16-byte aligned");
  const int64_t strides[] = {q_nope_user_stride, q_nope_head_stride, q_rope_user_stride, q_rope_head_stride, latent_user_stride,
                             rope_user_stride, w_uk_head_stride, w_uv_head_stride};
  for (int64_t s : strides) TTPA_REQUIRE(s % 8 == 0, "latent step: strides must be multiples of 8 elements");
  TTPA_REQUIRE(out_user_stride % 4 == 0 && out_head_stride % 4 == 0, "latent step: out strides must be multiples of 4 elements");
  // one of a weight's two inner dimensions is contiguous, the other's stride whole 16-byte pieces
  const bool uk_columns = w_uk_column_stride != 1, uv_columns = w_uv_column_stride != 1;
  const int64_t uk_ld = uk_columns ? w_uk_column_stride : w_uk_row_stride, uv_ld = uv_columns ? w_uv_column_stride : w_uv_row_stride;
  TTPA_REQUIRE((!uk_columns || w_uk_row_stride == 1) && (!uv_columns || w_uv_row_stride == 1),
               "latent step: the rows or the columns of a weight must be contiguous");
  TTPA_REQUIRE(uk_ld % 8 == 0 && uv_ld % 8 == 0, "latent step: strides must be multiples of 8 elements");
  TTPA_REQUIRE(uk_ld > 0 && uk_ld < (1 << 24) && uv_ld > 0 && uv_ld < (1 << 24), "latent step: weight row stride out of range");
  TTPA_REQUIRE(heads <= 65535 && (users + kUsers - 1) / kUsers <= 65535, "latent step: too many heads or users for one launch");
  const size_t need = ttpa_latent_decode_step_workspace_bytes(users, heads);
  if (need == 0) return fail(TTPA_ERR_UNSUPPORTED, "latent step: %d heads are not built", heads);
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 255u))
    return fail(TTPA_ERR_WORKSPACE, "latent step: workspace of %zu bytes (256-byte aligned) required, got %zu", need, workspace_bytes);
  const size_t attn = align256(ttpa_paged_mla_decode_workspace_bytes(users, heads, 1, kLatent));
  StepArgs a;
  a.q_nope = static_cast<const uint16_t *>(q_nope), a.qn_us = q_nope_user_stride, a.qn_hs = q_nope_head_stride;
  a.q_rope = static_cast<const uint16_t *>(q_rope), a.qr_us = q_rope_user_stride, a.qr_hs = q_rope_head_stride;
  a.latent = static_cast<const uint16_t *>(latent), a.latent_us = latent_user_stride;
  a.rope = static_cast<const uint16_t *>(rope), a.rope_us = rope_user_stride;
  a.w_uk = static_cast<const uint16_t *>(w_uk), a.uk_hs = w_uk_head_stride, a.uk_ld = uk_ld;
  a.w_uv = static_cast<const uint16_t *>(w_uv), a.uv_hs = w_uv_head_stride, a.uv_ld = uv_ld;
  a.q_lat = reinterpret_cast<uint16_t *>(static_cast<unsigned char *>(workspace) + attn);
  a.o_lat = reinterpret_cast<uint16_t *>(reinterpret_cast<unsigned char *>(a.q_lat) + align256((size_t)users * heads * kRow * 2));
  a.out = static_cast<uint16_t *>(out), a.out_us = out_user_stride, a.out_hs = out_head_stride;
  a.cache = static_cast<uint16_t *>(cache);
  a.pt = page_table, a.pt_rs = page_table_row_stride, a.pos = cur_pos, a.pos_i64 = cur_pos_is_i64;
  a.users = users, a.heads = heads, a.bs = block_size, a.w = table_width, a.nb = num_blocks;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 query_grid(kLatent / 128, (unsigned)heads, (unsigned)((a.users + kUsers - 1) / kUsers)), value_grid(kValue / 32, (unsigned)heads, lay_out_tiles(a));
  if (uk_columns) latent_query_kernel<true><<<query_grid, dim3(256), 0, st>>>(a);
  else latent_query_kernel<false><<<query_grid, dim3(256), 0, st>>>(a);
  if (int rc = check_launch("latent_decode_step (query)")) return rc;
  if (int rc = ttpa_paged_mla_decode(a.o_lat, (int64_t)heads * kLatent, kLatent, a.q_lat, (int64_t)heads * kRow, kRow, cache, nullptr,
                                     page_table, page_table_row_stride, cur_pos, cur_pos_is_i64, users, heads, 1, kRow, kLatent,
                                     block_size, table_width, num_blocks, scale, nullptr, workspace, attn, stream))
    return rc;
  if (uv_columns) latent_value_kernel<true><<<value_grid, dim3(256), 0, st>>>(a);
  else latent_value_kernel<false><<<value_grid, dim3(256), 0, st>>>(a);
  return check_launch("latent_decode_step (value)");
}

// Prompts of up to this many tokens are absorbed: their error against 64 bits is smaller there than expanded (16 heads, 32 / 64
// tokens 2.851e-3 / 2.975e-3 against 2.871e-3 / 2.993e-3; 96 / 512 tokens 3.062e-3 / 3.336e-3 against 3.056e-3 / 3.305e-3).
static constexpr int kAbsorbedTokens = 64;

extern "C" int64_t ttpa_latent_prompt_workspace_bytes(int32_t users, int32_t heads, int32_t seq_len) {
  if (users <= 0 || heads <= 0 || seq_len <= 0) return 0;
  const size_t rows = (size_t)users * seq_len, row = (size_t)heads * rows * 2;
  if (seq_len <= kAbsorbedTokens) return (int64_t)(align256(rows * kRow * 2) + align256(row * kRow) + align256(row * kLatent));
  return (int64_t)(2 * align256(row * 128));
}

extern "C" int ttpa_latent_prompt(void *out, int64_t out_token_stride, int64_t out_head_stride, const void *q_nope,
                                  int64_t q_nope_token_stride, int64_t q_nope_head_stride, const void *q_rope,
                                  int64_t q_rope_token_stride, int64_t q_rope_head_stride, const void *latent,
                                  int64_t latent_token_stride, const void *rope, int64_t rope_token_stride, const void *w_uk,
                                  int64_t w_uk_head_stride, int64_t w_uk_row_stride, int64_t w_uk_column_stride,
                                  const void *w_uv, int64_t w_uv_head_stride, int64_t w_uv_row_stride,
                                  int64_t w_uv_column_stride, void *cache, const int32_t *page_table,
                                  int64_t page_table_row_stride, int32_t users, int32_t table_rows, int32_t heads,
                                  int32_t seq_len, int32_t block_size, int32_t table_width, int32_t num_blocks, float scale,
                                  void *workspace, int64_t workspace_bytes, void *stream) {
  TTPA_REQUIRE(out && q_nope && q_rope && latent && rope && w_uk && w_uv, "null pointer argument");
  TTPA_REQUIRE(users > 0 && heads > 0 && seq_len > 0 && seq_len % 32 == 0, "latent prompt: bad users, heads or tokens");
  TTPA_REQUIRE(!cache || (page_table && table_rows > 0 && block_size > 0 && table_width > 0 && num_blocks > 0 &&
                          (int64_t)seq_len <= (int64_t)table_width * block_size),
               "latent prompt: %d tokens do not fit the page table", seq_len);
  TTPA_REQUIRE(aligned16(q_nope) && aligned16(q_rope) && aligned16(latent) && aligned16(rope) && aligned16(w_uk) && aligned16(w_uv) &&
                   aligned16(cache) && aligned16(out),
               "latent prompt: operands must be 16-byte aligned");
  const int64_t strides[] = {out_token_stride, out_head_stride, q_nope_token_stride, q_nope_head_stride, q_rope_token_stride, q_rope_head_stride,
                             latent_token_stride, rope_token_stride, w_uk_head_stride, w_uv_head_stride};
  for (int64_t s : strides) TTPA_REQUIRE(s % 8 == 0, "latent prompt: strides must be multiples of 8 elements");
  const bool uk_columns = w_uk_column_stride != 1, uv_columns = w_uv_column_stride != 1;
  const int64_t uk_ld = uk_columns ? w_uk_column_stride : w_uk_row_stride, uv_ld = uv_columns ? w_uv_column_stride : w_uv_row_stride;
  TTPA_REQUIRE((!uk_columns || w_uk_row_stride == 1) && (!uv_columns || w_uv_row_stride == 1),
               "latent prompt: the rows or the columns of a weight must be contiguous");
  TTPA_REQUIRE(uk_ld % 8 == 0 && uv_ld % 8 == 0 && uk_ld > 0 && uk_ld < (1 << 23) && uv_ld > 0 && uv_ld < (1 << 23) &&
                   latent_token_stride > 0 && latent_token_stride < (1 << 23),
               "latent prompt: row strides must be multiples of 8 elements below 2^23");
  const int64_t rows = (int64_t)users * seq_len, token_tiles = (rows + kExpTokens - 1) / kExpTokens;
  TTPA_REQUIRE(heads <= 65535 && rows <= (int64_t)65535 * kUsers && token_tiles * 2 * heads + rows < (int64_t)1 << 31,
               "latent prompt: too many heads or tokens for one launch");
  const int64_t need = ttpa_latent_prompt_workspace_bytes(users, heads, seq_len);
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 255u))
    return fail(TTPA_ERR_WORKSPACE, "latent prompt: workspace of %lld bytes (256-byte aligned) required, got %lld", (long long)need,
                (long long)workspace_bytes);
  unsigned char *ws = static_cast<unsigned char *>(workspace);
  ExpandArgs e{};
  StepArgs &a = e.s;
  a.q_nope = static_cast<const uint16_t *>(q_nope), a.qn_us = q_nope_token_stride, a.qn_hs = q_nope_head_stride;
  a.q_rope = static_cast<const uint16_t *>(q_rope), a.qr_us = q_rope_token_stride, a.qr_hs = q_rope_head_stride;
  a.latent = static_cast<const uint16_t *>(latent), a.latent_us = latent_token_stride;
  a.rope = static_cast<const uint16_t *>(rope), a.rope_us = rope_token_stride;
  a.w_uk = static_cast<const uint16_t *>(w_uk), a.uk_hs = w_uk_head_stride, a.uk_ld = uk_ld;
  a.w_uv = static_cast<const uint16_t *>(w_uv), a.uv_hs = w_uv_head_stride, a.uv_ld = uv_ld;
  a.out = static_cast<uint16_t *>(out), a.out_us = out_token_stride, a.out_hs = out_head_stride;
  a.cache = static_cast<uint16_t *>(cache), a.pt = page_table, a.pt_rs = page_table_row_stride;
  a.users = (int)rows, a.heads = heads, a.bs = block_size, a.w = table_width, a.nb = num_blocks;
  a.seq = seq_len, a.table_rows = table_rows;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (seq_len > kAbsorbedTokens) {
    e.k = reinterpret_cast<uint16_t *>(ws), e.v = reinterpret_cast<uint16_t *>(ws + align256((size_t)rows * heads * 256));
    e.uk_rows = !uk_columns, e.uv_rows = uv_columns;
    e.items = (int)(token_tiles * 2 * heads);
    const bool shared = (e.items > 256 && e.items < 480) || e.items >= 800;  // (of 512 places, two on a CU: ExpandShape)
    if (int rc = shared ? launch_expand<ExpandShape<64, 2>>(e, st) : launch_expand<ExpandShape<32, 4>>(e, st)) return rc;
    const int64_t hd = (int64_t)heads * 128, sl = seq_len;
    return ttpa_split_key_prefill(out, sl * out_token_stride, out_head_stride, out_token_stride, q_nope, sl * q_nope_token_stride,
                                  q_nope_head_stride, q_nope_token_stride, q_rope, sl * q_rope_token_stride, q_rope_head_stride,
                                  q_rope_token_stride, e.k, sl * hd, 128, hd, rope, sl * rope_token_stride, 0, rope_token_stride, e.v,
                                  sl * hd, 128, hd, users, heads, heads, seq_len, scale, stream);
  }
  a.k_lat = reinterpret_cast<uint16_t *>(ws);
  a.q_lat = reinterpret_cast<uint16_t *>(ws + align256((size_t)rows * kRow * 2));
  a.o_lat = reinterpret_cast<uint16_t *>(reinterpret_cast<unsigned char *>(a.q_lat) + align256((size_t)rows * heads * kRow * 2));
  const dim3 query_grid(kLatent / 128, (unsigned)heads, (unsigned)((a.users + kUsers - 1) / kUsers)), value_grid(kValue / 32, (unsigned)heads, lay_out_tiles(a));
  if (uk_columns) latent_query_kernel<true, true><<<query_grid, dim3(256), 0, st>>>(a);
  else latent_query_kernel<false, true><<<query_grid, dim3(256), 0, st>>>(a);
  if (int rc = check_launch("latent_prompt (query)")) return rc;
  const int64_t ql = (int64_t)heads * kRow, ol = (int64_t)heads * kLatent;
  if (int rc = ttpa_latent_prefill(a.o_lat, seq_len * ol, kLatent, ol, a.q_lat, seq_len * ql, kRow, ql, a.k_lat, (int64_t)seq_len * kRow, 0, kRow,
                                   nullptr, 0, 0, 0, users, heads, 1, seq_len, kRow, kLatent, 1, scale, stream))
    return rc;
  if (uv_columns) latent_value_kernel<true><<<value_grid, dim3(256), 0, st>>>(a);
  else latent_value_kernel<false><<<value_grid, dim3(256), 0, st>>>(a);
  return check_launch("latent_prompt (value)");
}
