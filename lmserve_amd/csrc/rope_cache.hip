// Rotary position embedding fused with the K/V write (gfx950).
//
// In the reference's attention layer the rotation of Q and K runs as its own
// launch immediately before the cache write, on the same K tensor. Here a
// workgroup belongs to ONE token (so position, cos/sin row and cache slot are
// workgroup-uniform): its lanes rotate Q and K in fp32 with a single rounding
// to the storage type and, when a cache is given, store the rotated K and the V
// row straight into the token's slot. K is read once and V never takes a
// separate launch. Without a cache the kernel is the plain rotation.
//
// Vectors are 16 bytes (8 bf16/fp16 or 4 fp32 elements); a "pair-vector" is the
// x half and the y half of the same rotation lanes of one head.

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <new>

#include "common.h"
#include "device.h"
#include "kvcache.h"
#include "kvcache_experimental.h"

namespace kvc {
RopeTuning g_rope_tune;
}

namespace {

using kvc::fail;
using kvc::log2_exact;
using kvc::OutRow;
using kvc::u32x4;

constexpr int kThreads = 256;
constexpr int kMaxRotaryDim = 512;  // at most 64 pair-vectors a head (fp32): what the division by pairs_magic relies on

// ---- storage types ---------------------------------------------------------
struct BF16 {
  static constexpr int kBytes = 2;
  static __device__ __forceinline__ float load(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
  // Round to nearest, ties to even, through the native conversion: gfx950 has a
  // packed f32 -> bf16 convert instruction, which the compiler selects for this.
  static __device__ __forceinline__ uint16_t store(float f) {
    return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
  }
  static __device__ __forceinline__ uint32_t store2(float lo, float hi) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
};
struct F16 {
  static constexpr int kBytes = 2;
  static __device__ __forceinline__ float load(uint16_t b) { return __half2float(__ushort_as_half(b)); }
  static __device__ __forceinline__ uint16_t store(float f) { return __half_as_ushort(__float2half_rn(f)); }
  static __device__ __forceinline__ uint32_t store2(float lo, float hi) {
    return (uint32_t)store(lo) | ((uint32_t)store(hi) << 16);
  }
};
struct F32 {
  static constexpr int kBytes = 4;
};

// one 16-byte pair-vector in fp32 with one rounding: ox = x cos - y sin, oy = y cos + x sin; contracted by hand, the
// own half's product in the fma: the same bits in every kernel
template <typename T>
struct Vec {
  static __device__ __forceinline__ void rotate(u32x4 x, u32x4 y, u32x4 cx, u32x4 cy, u32x4 sx, u32x4 sy,
                                                u32x4& ox, u32x4& oy) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float o[2][2];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const auto f = [&](u32x4 v) { return T::load((uint16_t)(w ? v[i] >> 16 : v[i] & 0xffffu)); };
        o[0][w] = __builtin_fmaf(f(x), f(cx), -(f(y) * f(sx)));
        o[1][w] = __builtin_fmaf(f(y), f(cy), f(x) * f(sy));
      }
      ox[i] = T::store2(o[0][0], o[0][1]);
      oy[i] = T::store2(o[1][0], o[1][1]);
    }
  }
  // one 16-byte vector of either half, `other` the same lanes of the other half: own cos -+ other sin, the minus by
  // `flip` in the sign bits of the x half; contracted as `rotate` is
  static constexpr uint32_t kSign = 0x80008000u;
  static __device__ __forceinline__ u32x4 rotate_one(u32x4 own, u32x4 other, u32x4 c, u32x4 s, uint32_t flip) {
    u32x4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float r[2];
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const auto f = [&](uint32_t v) { return T::load((uint16_t)(w ? v >> 16 : v & 0xffffu)); };
        r[w] = __builtin_fmaf(f(own[i]), f(c[i]), f(other[i]) * f(s[i] ^ flip));
      }
      out[i] = T::store2(r[0], r[1]);
    }
    return out;
  }
  // one element
  typedef uint16_t Word;
  static __device__ __forceinline__ float wide(Word w) { return T::load(w); }
  static __device__ __forceinline__ Word narrow(float f) { return T::store(f); }
};
template <>
struct Vec<F32> {
  static __device__ __forceinline__ void rotate(u32x4 x, u32x4 y, u32x4 cx, u32x4 cy, u32x4 sx, u32x4 sy,
                                                u32x4& ox, u32x4& oy) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const auto f = [&](u32x4 v) { return __uint_as_float(v[i]); };
      ox[i] = __float_as_uint(__builtin_fmaf(f(x), f(cx), -(f(y) * f(sx))));
      oy[i] = __float_as_uint(__builtin_fmaf(f(y), f(cy), f(x) * f(sy)));
    }
  }
  static constexpr uint32_t kSign = 0x80000000u;
  static __device__ __forceinline__ u32x4 rotate_one(u32x4 own, u32x4 other, u32x4 c, u32x4 s, uint32_t flip) {
    u32x4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[i] = __float_as_uint(__builtin_fmaf(__uint_as_float(own[i]), __uint_as_float(c[i]),
                                              __uint_as_float(other[i]) * __uint_as_float(s[i] ^ flip)));
    return out;
  }
  typedef uint32_t Word;
  static __device__ __forceinline__ float wide(Word w) { return __uint_as_float(w); }
  static __device__ __forceinline__ Word narrow(float f) { return __float_as_uint(f); }
};

struct RopeArgs {
  const char* query;
  const char* key;
  const char* value;       // null without a cache
  char* query_out;
  char* key_out;           // may be null when a cache takes the rotated K
  const void* positions;   // rotation positions; with page-table addressing also the KV positions
  int pos_bytes;
  const char* cos_sin_cache;  // [max_position, 2*rotary_dim]: cos | sin
  int64_t max_position;
  uint32_t num_heads, num_kv_heads, head_dim, rotary_dim;
  int64_t q_token_stride, k_token_stride, v_token_stride;     // bytes
  int64_t qo_token_stride, ko_token_stride;                   // bytes
  // cache side (key_cache == null: plain rotation)
  char* key_cache;
  char* value_cache;
  const void* slot_mapping;
  int slot_bytes;
  const int32_t* batch_indices;  // non-null: page-table addressing
  const int32_t* kv_indices;
  const int32_t* kv_indptr;
  int64_t batch_size, num_kv_indices;
  int64_t block_size;
  int bs_shift;
  int64_t cache_block_stride, cache_slot_stride;  // bytes
  int64_t num_cache_blocks;
  uint32_t groups_per_token;  // workgroups per token
  uint32_t threads;           // lanes of a workgroup
  // vector kernels
  uint32_t lanes_per_token;   // lanes that have work
  uint32_t pairs_per_head;    // pair-vectors of one head
  uint32_t split;             // a lane's head is lane / split: pairs_per_head, or the vectors of a head (rows kernel)
  uint32_t split_magic;       // ceil(2^32 / split): lane / split = mulhi(lane, magic); 0 where that is not exact
  uint32_t head_step;         // rows kernel: heads between a lane's two
  uint32_t v_items;           // 16-byte vectors of the token's V row (0 without a cache)
  uint32_t cache_nt;          // pair form: cache rows by non-temporal stores
};

// The same in 128 bytes, for the kernels that take the index build's types and rows of aligned vectors; byte strides
// and counts that do not fit send a call to the general form. A launch's arguments are written to memory beyond the
// host link. What that costs the host hangs on a state of the host that changes from machine to machine and within
// minutes. Launches of one layer back to back, RopeArgs with the 256 bytes of launch geometry that a kernel takes along once
// it reads blockDim, and these, us each (32 layers of 256 tokens x 32 + 8 heads x 128; medians of 16 runs in turn): 4.4 and
// 3.6 where the step at 128 bytes showed most, 4.12 and 4.15, 3.18 and 3.14, and 2.45 both. On the device by slot the short
// form is 1 % ahead (rows form 3 to 5), and several layers in one launch gain most (64 tokens x 28 layers of 28 + 4 x 128 4.56
// and 4.30, 256 x 16 of 32 + 8 x 64 6.4 and 5.9, 256 x 80 of 8 + 1 x 128, which takes one launch instead of two, 16.8 and 12.8).
struct RopeLean {
  const char *query, *key, *value;
  char *query_out, *key_out, *key_cache, *value_cache;
  const void* positions;
  const char* cos_sin_cache;
  const void* slot_mapping;
  uint32_t q_token_stride, k_token_stride, v_token_stride, qo_token_stride, ko_token_stride;  // bytes
  uint32_t max_position;
  uint32_t cache_block_stride, cache_slot_stride;  // bytes
  uint32_t num_cache_blocks;
  uint32_t split_magic;
  uint16_t num_heads, num_kv_heads;
  uint8_t pairs_per_head, vecs_per_head, bs_shift;
  uint8_t shape;  // cache_nt, then the workgroup's wavefronts
};
static_assert(sizeof(RopeLean) == 128, "where a launch's arguments begin to cost more");
struct RopeLeanPages : RopeLean {
  const int32_t *batch_indices, *kv_indices, *kv_indptr;
  uint32_t batch_size, num_kv_indices;
};

// One layer's buffers, as RopeArgs names them
struct RopeLayer {
  const char *query, *key, *value;
  char *query_out, *key_out, *key_cache, *value_cache;
};

// How a token finds its cache slot: not at all (plain rotation), through a slot
// mapping, or through the page table.
enum Addressing : int { kNoCache, kSlots, kPages };

// The kernels of rows of aligned 16-byte vectors, and the one of all other rows
enum VectorForm {
  kElements = KVC_ROPE_ELEMENTS, kPairs = KVC_ROPE_PAIRS, kRows = KVC_ROPE_ROWS, kOwner = KVC_ROPE_OWNER,
  kOwnerTail = KVC_ROPE_OWNER_TAIL
};

template <Addressing ADDR> struct LeanOf { using type = RopeLean; };
template <> struct LeanOf<kPages> { using type = RopeLeanPages; };

// Lanes of a token that have work
template <typename I>
__host__ __device__ __forceinline__ I lanes_of(VectorForm form, I heads, I kv_heads, I pairs, I vecs, bool cache) {
  if (form == kRows) return (heads + (cache ? 2 * kv_heads : kv_heads) + 1) / 2 * vecs;
  const I pair_lanes = (heads + kv_heads) * pairs;
  if (form != kOwnerTail) return pair_lanes;
  const I extras = (cache ? kv_heads * vecs : 0) + (heads + kv_heads) * (vecs - 2 * pairs);
  return pair_lanes > (extras + 1) / 2 ? pair_lanes : (extras + 1) / 2;
}

// What a kernel of this form reads of RopeArgs, the rest left alone
template <typename T, Addressing ADDR, VectorForm FORM>
__device__ __forceinline__ RopeArgs from_lean(const typename LeanOf<ADDR>::type& l) {
  RopeArgs a;
  a.query = l.query; a.key = l.key; a.value = l.value;
  a.query_out = l.query_out; a.key_out = l.key_out; a.key_cache = l.key_cache; a.value_cache = l.value_cache;
  a.positions = l.positions; a.cos_sin_cache = l.cos_sin_cache; a.max_position = l.max_position;
  a.num_heads = l.num_heads; a.num_kv_heads = l.num_kv_heads;
  a.head_dim = l.vecs_per_head * (16u / T::kBytes);
  a.rotary_dim = l.pairs_per_head * (32u / T::kBytes);
  a.q_token_stride = l.q_token_stride; a.k_token_stride = l.k_token_stride; a.v_token_stride = l.v_token_stride;
  a.qo_token_stride = l.qo_token_stride; a.ko_token_stride = l.ko_token_stride;
  a.slot_mapping = l.slot_mapping;
  if constexpr (ADDR == kPages) {
    a.batch_indices = l.batch_indices; a.kv_indices = l.kv_indices; a.kv_indptr = l.kv_indptr;
    a.batch_size = l.batch_size; a.num_kv_indices = l.num_kv_indices;
  }
  a.bs_shift = l.bs_shift;
  a.cache_block_stride = l.cache_block_stride; a.cache_slot_stride = l.cache_slot_stride;
  a.num_cache_blocks = l.num_cache_blocks;
  a.threads = (uint32_t)(l.shape >> 1) * 64;
  a.lanes_per_token = lanes_of<uint32_t>(FORM, l.num_heads, l.num_kv_heads, l.pairs_per_head, l.vecs_per_head, ADDR != kNoCache);
  a.pairs_per_head = l.pairs_per_head;
  a.split = FORM == kRows ? l.vecs_per_head : l.pairs_per_head;
  a.split_magic = l.split_magic;
  a.head_step = ((uint32_t)l.num_heads + (ADDR != kNoCache ? 2 : 1) * (uint32_t)l.num_kv_heads + 1) / 2;
  a.v_items = ADDR == kNoCache ? 0 : (uint32_t)l.num_kv_heads * l.vecs_per_head;
  a.cache_nt = l.shape & 1;
  return a;
}

// Entry t of an int32 or int64 array (width in bytes). Two loads side by side and no
// branch: a branch on the width makes the scalar unit wait for the value inside it.
__device__ __forceinline__ int64_t index_of(const void* array, int width, uint32_t t) {
  const int32_t words = width >> 2;
  const int32_t* p = reinterpret_cast<const int32_t*>(array) + (int64_t)t * words;
  const int32_t lo = p[0], hi = p[words - 1];
  return ((int64_t)(words == 2 ? hi : lo >> 31) << 32) | (uint32_t)lo;
}

// Byte offset of token t's slot from the start of a cache plane, or -1 where the
// write skips the token. Uniform over the workgroup: scalar loads. FAST: int32
// positions, int64 slots and a block size that is a power of two, as the index
// build makes them; the other form handles either width and carries 64-bit
// divisions (a decode launch of 256 tokens, rows in cache, takes 2.65 us with the widths
// fixed, 2.73 with both words loaded side by side, 3.4 with the divisions as well).
template <Addressing ADDR, bool FAST>
__device__ __forceinline__ int64_t slot_offset(const RopeArgs& a, uint32_t t, int64_t pos) {
  if constexpr (ADDR == kNoCache) return -1;
  int64_t blk = -1, off = 0;
  if constexpr (ADDR == kPages) {
    // an index that is out of range is read as 0 (the host has looked that there are requests and pages): a branch
    // per check makes each load wait for the one before
    const int64_t b = a.batch_indices[t];
    const bool known = b >= 0 && b < a.batch_size;
    const int64_t bc = known ? b : 0, begin = a.kv_indptr[bc], end = a.kv_indptr[bc + 1];
    const int64_t pg = FAST ? (pos >> a.bs_shift) : pos / a.block_size;
    off = pos - (FAST ? pg << a.bs_shift : pg * a.block_size);
    const int64_t it = begin + pg;
    const bool ok = known && it >= 0 && it < end && it < a.num_kv_indices;
    const int64_t page = a.kv_indices[ok ? it : 0];
    if (ok) blk = page;
  } else {
    const int64_t s = FAST ? reinterpret_cast<const int64_t*>(a.slot_mapping)[t] : index_of(a.slot_mapping, a.slot_bytes, t);
    if (s >= 0) {
      blk = FAST ? (s >> a.bs_shift) : s / a.block_size;
      off = s - (FAST ? blk << a.bs_shift : blk * a.block_size);
    }
  }
  if (blk < 0 || blk >= a.num_cache_blocks) return -1;
  return blk * a.cache_block_stride + off * a.cache_slot_stride;
}

template <bool NT>
__device__ __forceinline__ u32x4 ld16(const char* p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  else return *reinterpret_cast<const u32x4*>(p);
}
// 16 bytes of a cos/sin row, which may start at any element (a table that is a view): the same one load. 2048 tokens
// x 40 heads x 128 with the cache: 9.3 us where the table is 16-byte aligned, 10.0 where to 4 bytes, 11.4 where to 2;
// an element at a time, rows and all, 37.3.
typedef u32x4 __attribute__((aligned(2))) u32x4_at_any_element;
__device__ __forceinline__ u32x4 ld16_cos_sin(const char* p) {
  return *reinterpret_cast<const u32x4_at_any_element*>(p);
}
// lane / split, the magic uniform. Where split is pairs_per_head the magic is 0 for 1 alone, and the kernels do without
// the division.
__device__ __forceinline__ uint32_t head_of_pair(const RopeArgs& a, uint32_t lane) {
  return a.split_magic ? __umulhi(lane, a.split_magic) : lane;
}
__device__ __forceinline__ uint32_t head_of_lane(const RopeArgs& a, uint32_t lane) {
  return a.split_magic ? __umulhi(lane, a.split_magic) : lane / a.split;
}

// Whole heads rotated, halves of whole 64-byte pieces. A lane owns ONE pair-vector of one
// Q or K head and carries a V vector along, so a token is as few wavefronts as its
// pair-vectors need (a V row of its own lanes costs 8 heads x 128 a sixth wavefront, 4
// heads a fifth). blockIdx = (group, token).
// What bounds it: at decode sizes the chain launch -> position -> cos/sin row ->
// store and the instructions on it; at prefill sizes HBM. Hence
//   - the lane's own four 16-byte pieces of the cos/sin row go straight to
//     registers; staging the row in LDS as fp32 for all heads puts an LDS write, a
//     barrier and 32 LDS words per lane on that chain. Two and four heads per lane
//     share the pieces and lose more in wavefronts in flight (a fifth and two fifths
//     more time at decode sizes, a tenth at 2048 tokens);
//   - nothing waits for the position before the Q, K and V loads are issued;
//   - an instantiation holds only the code its launch needs: every addressing form
//     and 64-bit divisions in one kernel cost a decode launch 15 %.
// query_out is stored at device scope, the cache rows the same, and non-temporal beyond
// 3 MiB of them. What plain stores leave dirty in the L2s is written back when the launch
// ends, and a reader, mostly on another XCD, finds it in the last-level cache either way.
// Launch of a recorded step alone, and with a copy of query_out behind it, plain and
// non-temporal stores -> these (us): 256 tokens x 40 heads x 128 3.10 -> 2.80 and 5.55 ->
// 5.20; 1024 of those 5.87 -> 5.38 and 9.57 -> 9.20; 2048 x 32 x 128 8.45 -> 7.74 and 13.72
// -> 13.13; 2048 x 72 x 128 17.15 -> 16.61 and 27.44 -> 26.79; 8192 of those 59.4 -> 58.1
// (5.8 TB/s) and 124 -> 120.5. Non-temporal query_out is faster still alone and costs its
// reader more (1024 tokens 5.21 and 10.07; 2048 x 72 14.24 and 30.02). So do few cache rows,
// non-temporal -> not, alone and with a gather of the rows behind the launch, in pools that no
// cache holds: 1 token of 28 + 4 heads x 128 2.17 -> 2.19 and 4.46 -> 4.17, 512 2.78 -> 2.77
// and 5.69 -> 5.40, 1024 (2 MiB) 4.79 -> 4.53 and 7.64 -> 6.95; 2048 (4 MiB) 7.24 -> 7.19 and
// 10.6 -> 10.8, of 32 + 8 x 64 5.55 -> 5.80 and 8.84 -> 8.78; 4096 of 32 + 32 x 128 34.7 -> 39.5
// alone. Stores at device scope of pieces that are no whole 64 bytes lose (2048 x 15 x 96 in
// bf16, halves of 96 bytes, 4.68 -> 5.16): such heads, and outputs that start within 64 bytes,
// go to the rows kernel.
// NTL: non-temporal loads, bit 0 for the K and V rows, bit 1 for the Q rows; by size, see run_rope.
template <typename T, Addressing ADDR, int NTL>
__device__ __forceinline__ void rope_pairs_lane(const RopeArgs& a, const RopeLayer p) {
  constexpr uint32_t E = T::kBytes;
  const uint32_t t = blockIdx.y;
  const uint32_t lane = blockIdx.x * a.threads + threadIdx.x;
  if (lane >= a.lanes_per_token) return;
  const int64_t pos = reinterpret_cast<const int32_t*>(a.positions)[t];

  const uint32_t half = (a.rotary_dim >> 1) * E;  // bytes
  const uint32_t h = head_of_pair(a, lane);
  const uint32_t pv = (lane - h * a.split) * 16;
  const bool is_k = h >= a.num_heads;
  const uint32_t head_off = (is_k ? h - a.num_heads : h) * a.head_dim * E + pv;
  u32x4 x, y;
  if (NTL == 1 || NTL == 2) {
    if (is_k) {
      const char* in = p.key + (int64_t)t * a.k_token_stride + head_off;
      x = ld16<(NTL & 1) != 0>(in);
      y = ld16<(NTL & 1) != 0>(in + half);
    } else {
      const char* in = p.query + (int64_t)t * a.q_token_stride + head_off;
      x = ld16<(NTL & 2) != 0>(in);
      y = ld16<(NTL & 2) != 0>(in + half);
    }
  } else {
    const char* in = (is_k ? p.key + (int64_t)t * a.k_token_stride : p.query + (int64_t)t * a.q_token_stride) + head_off;
    x = ld16<NTL != 0>(in);
    y = ld16<NTL != 0>(in + half);
  }
  const bool has_v = ADDR != kNoCache && lane < a.v_items;
  u32x4 v = {};
  if (has_v) v = ld16<(NTL & 1) != 0>(p.value + (int64_t)t * a.v_token_stride + lane * 16);

  if (pos < 0 || pos >= a.max_position) return;  // no cos/sin row: the token is left alone
  const char* row = a.cos_sin_cache + pos * (int64_t)(4 * half) + pv;
  const u32x4 cos_x = ld16_cos_sin(row), cos_y = ld16_cos_sin(row + half), sin_x = ld16_cos_sin(row + 2 * half),
              sin_y = ld16_cos_sin(row + 3 * half);
  const int64_t slot = slot_offset<ADDR, true>(a, t, pos);

  u32x4 ox, oy;
  Vec<T>::rotate(x, y, cos_x, cos_y, sin_x, sin_y, ox, oy);
  const uint32_t kv_bytes = a.num_kv_heads * a.head_dim * E;
  if (!is_k) {
    const OutRow out(p.query_out + (int64_t)t * a.qo_token_stride, a.num_heads * a.head_dim * E);
    out.store<kvc::kThrough>(head_off, ox);
    out.store<kvc::kThrough>(head_off + half, oy);
  } else {
    if (p.key_out) {
      const OutRow out(p.key_out + (int64_t)t * a.ko_token_stride, kv_bytes);
      out.store<kvc::kThrough>(head_off, ox);
      out.store<kvc::kThrough>(head_off + half, oy);
    }
    if (ADDR != kNoCache && slot >= 0) {
      const OutRow out(p.key_cache + slot, kv_bytes);
      if (a.cache_nt) {
        out.store<kvc::kThroughNt>(head_off, ox);
        out.store<kvc::kThroughNt>(head_off + half, oy);
      } else {
        out.store<kvc::kThrough>(head_off, ox);
        out.store<kvc::kThrough>(head_off + half, oy);
      }
    }
  }
  if (has_v && slot >= 0) {
    const OutRow out(p.value_cache + slot, kv_bytes);
    if (a.cache_nt) out.store<kvc::kThroughNt>(lane * 16, v);
    else out.store<kvc::kThrough>(lane * 16, v);
  }
}

// Every other shape of aligned rows that are written elsewhere than where they are read:
// heads rotated in part, halves that are no whole 64-byte pieces, more V vectors than
// pair-vectors, other index types. A lane owns the same 16-byte vector of two heads (Q, then K, then V heads), so the lanes write the rows out in
// order, whole lines whatever the halves are; its other half's vector is a second load, from the
// first-level cache. With the pair form, a lane's unrotated vectors carried along, a
// partial rotation wrote pieces of 32 and 96 bytes. Launch of a recorded step alone, and
// with a copy of query_out behind it, that form -> this (us): 838 tokens x 40 heads x 80, 32
// rotated, 4.99 -> 3.99 and 8.00 -> 7.12; 8192 of those 33.7 -> 23.7 and 43.5 -> 35.0; 256 3.49 ->
// 2.93; 2048 x 15 x 96 in bf16 4.65 -> 4.25 and 7.74 -> 7.28; 2048 x 40 x 128, 64 rotated, 9.6 -> 9.7
// and 15.3 -> 15.9, 300 of those 3.80 -> 3.13, 8192 38.5 -> 35.9 and 61.2 -> 59.5. One head per lane
// is 5 to 9 % slower at prefill sizes, three 2 to 7 %; the other half by shuffles is no
// faster than by the load.
template <typename T, Addressing ADDR, bool FAST, int NTL>
__device__ __forceinline__ void rope_rows_lane(const RopeArgs& a, const RopeLayer p) {
  constexpr uint32_t E = T::kBytes;
  constexpr int HEADS = 2;
  const uint32_t t = blockIdx.y;
  const uint32_t lane = blockIdx.x * a.threads + threadIdx.x;
  if (lane >= a.lanes_per_token) return;
  const int64_t pos = FAST ? (int64_t) reinterpret_cast<const int32_t*>(a.positions)[t] : index_of(a.positions, a.pos_bytes, t);

  const uint32_t h0 = head_of_lane(a, lane), v = lane - h0 * a.split, head_bytes = a.head_dim * E;
  const uint32_t hq = a.num_heads, hk = hq + a.num_kv_heads, heads = ADDR == kNoCache ? hk : hk + a.num_kv_heads;
  const bool first = v < a.pairs_per_head, rotates = v < 2 * a.pairs_per_head;
  const int32_t to_other = !rotates ? 0 : first ? (int32_t)a.pairs_per_head * 16 : -(int32_t)a.pairs_per_head * 16;
  const char* q_row = p.query + (int64_t)t * a.q_token_stride;
  const char* k_row = p.key + (int64_t)t * a.k_token_stride;
  const char* v_row = ADDR == kNoCache ? nullptr : p.value + (int64_t)t * a.v_token_stride;
  u32x4 own[HEADS], other[HEADS];
  uint32_t off[HEADS];
#pragma unroll
  for (int j = 0; j < HEADS; ++j) {
    const uint32_t h = min(h0 + j * a.head_step, heads - 1);  // a lane without a second head loads the last and stores none
    const bool is_q = h < hq, is_v = h >= hk;
    off[j] = (h - (is_q ? 0 : is_v ? hk : hq)) * head_bytes + v * 16;
    const char* in = (is_q ? q_row : is_v ? v_row : k_row) + off[j];
    if ((NTL == 1 || NTL == 2) && is_q != (NTL == 2)) {
      own[j] = ld16<false>(in);
      other[j] = ld16<false>(in + to_other);
    } else {
      own[j] = ld16<NTL != 0>(in);
      other[j] = ld16<NTL != 0>(in + to_other);
    }
  }

  if (pos < 0 || pos >= a.max_position) return;  // no cos/sin row: the token is left alone
  u32x4 c = {}, s = {};
  if (rotates) {
    const char* row = a.cos_sin_cache + pos * (int64_t)(2 * a.rotary_dim * E) + v * 16;
    c = ld16_cos_sin(row);
    s = ld16_cos_sin(row + a.rotary_dim * E);
  }
  const int64_t slot = slot_offset<ADDR, FAST>(a, t, pos);

  const uint32_t flip = first ? Vec<T>::kSign : 0u, kv_bytes = a.num_kv_heads * head_bytes;
#pragma unroll
  for (int j = 0; j < HEADS; ++j) {
    const uint32_t h = h0 + j * a.head_step;
    u32x4 out = own[j];
    if (rotates && h < hk) out = Vec<T>::rotate_one(own[j], other[j], c, s, flip);
    if (h < hq) {
      OutRow(p.query_out + (int64_t)t * a.qo_token_stride, hq * head_bytes).store<kvc::kThrough>(off[j], out);
    } else if (h < hk) {
      if (p.key_out) OutRow(p.key_out + (int64_t)t * a.ko_token_stride, kv_bytes).store<kvc::kThrough>(off[j], out);
      if (ADDR != kNoCache && slot >= 0) OutRow(p.key_cache + slot, kv_bytes).store<kvc::kThroughNt>(off[j], out);
    } else if (h < heads && slot >= 0) {
      OutRow(p.value_cache + slot, kv_bytes).store<kvc::kThroughNt>(off[j], out);
    }
  }
}

// Small launches of whole heads, and an output in its input's own rows: the pair form for every shape, since a lane of
// the rows kernel reads a vector that another lane overwrites. A lane owns both halves of a pair and carries vectors that pass through along: one of
// V, with TAIL up to two of V and of the heads' unrotated lanes. Bound as the pair form; plain stores, as its pieces
// are of any size. TAIL costs a launch without tails a tenth. us a launch of a recorded step, in place here and
// elsewhere by the rows kernel: 838 tokens x 40 heads x 80 in fp16, 32 rotated, 5.4 and 4.4, 8192 of those 30.1 and
// 21.8; 2048 x 15 x 96 in bf16 4.9 and 4.5, 256 of those 3.25 and 3.3.
template <typename T, Addressing ADDR, bool FAST, bool TAIL>
__device__ __forceinline__ void rope_owner_lane(const RopeArgs& a, const RopeLayer p) {
  constexpr uint32_t E = T::kBytes;
  const uint32_t t = blockIdx.y;
  const uint32_t lane = blockIdx.x * a.threads + threadIdx.x;
  if (lane >= a.lanes_per_token) return;
  const int64_t pos = FAST ? (int64_t) reinterpret_cast<const int32_t*>(a.positions)[t] : index_of(a.positions, a.pos_bytes, t);

  const uint32_t half = (a.rotary_dim >> 1) * E;  // bytes
  const uint32_t h = head_of_pair(a, lane);
  const uint32_t pv = (lane - h * a.split) * 16;
  const uint32_t heads = a.num_heads + a.num_kv_heads;
  const bool rotates = !TAIL || h < heads, is_k = h >= a.num_heads;
  const uint32_t head_off = (is_k ? h - a.num_heads : h) * a.head_dim * E + pv;
  const char* q_row = p.query + (int64_t)t * a.q_token_stride;
  const char* k_row = p.key + (int64_t)t * a.k_token_stride;
  u32x4 x = {}, y = {};
  if (rotates) {
    const char* in = (is_k ? k_row : q_row) + head_off;
    x = ld16<false>(in);
    y = ld16<false>(in + half);
  }
  enum Kind { kNone, kV, kTailQ, kTailK };
  constexpr int kCarried = TAIL ? 2 : 1;
  u32x4 carried[kCarried] = {};
  uint32_t carried_off[kCarried] = {};  // in the row it comes from and in the row it goes to
  Kind kind[kCarried];
#pragma unroll
  for (int j = 0; j < kCarried; ++j) {
    const uint32_t e = lane + j * a.lanes_per_token;
    kind[j] = kNone;
    if (ADDR != kNoCache && e < a.v_items) {
      kind[j] = kV;
      carried_off[j] = e * 16;
      carried[j] = ld16<false>(p.value + (int64_t)t * a.v_token_stride + carried_off[j]);
    } else if constexpr (TAIL) {
      const uint32_t tail_per_head = (a.head_dim - a.rotary_dim) * E / 16;
      if (e < a.v_items + heads * tail_per_head) {
        const uint32_t i = e - a.v_items, th = i / tail_per_head;
        const bool tk = th >= a.num_heads;
        kind[j] = tk ? kTailK : kTailQ;
        carried_off[j] = ((tk ? th - a.num_heads : th) * a.head_dim + a.rotary_dim) * E + (i - th * tail_per_head) * 16;
        carried[j] = ld16<false>((tk ? k_row : q_row) + carried_off[j]);
      }
    }
  }

  if (pos < 0 || pos >= a.max_position) return;  // no cos/sin row: the token is left alone
  u32x4 cos_x = {}, cos_y = {}, sin_x = {}, sin_y = {};
  if (rotates) {
    const char* row = a.cos_sin_cache + pos * (int64_t)(4 * half) + pv;
    cos_x = ld16_cos_sin(row);
    cos_y = ld16_cos_sin(row + half);
    sin_x = ld16_cos_sin(row + 2 * half);
    sin_y = ld16_cos_sin(row + 3 * half);
  }
  const int64_t slot = slot_offset<ADDR, FAST>(a, t, pos);

  const auto put = [](char* out, u32x4 v) { *reinterpret_cast<u32x4*>(out) = v; };
  const auto put_cache = [](char* out, u32x4 v) { __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out)); };
  if (rotates) {
    u32x4 ox, oy;
    Vec<T>::rotate(x, y, cos_x, cos_y, sin_x, sin_y, ox, oy);
    if (!is_k) {
      char* out = p.query_out + (int64_t)t * a.qo_token_stride + head_off;
      put(out, ox);
      put(out + half, oy);
    } else {
      if (p.key_out) {
        char* out = p.key_out + (int64_t)t * a.ko_token_stride + head_off;
        put(out, ox);
        put(out + half, oy);
      }
      if (ADDR != kNoCache && slot >= 0) {
        char* out = p.key_cache + slot + head_off;
        put_cache(out, ox);
        put_cache(out + half, oy);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kCarried; ++j) {
    if (kind[j] == kV) {
      if (slot >= 0) put_cache(p.value_cache + slot + carried_off[j], carried[j]);
    } else if (TAIL && kind[j] == kTailQ) {
      put(p.query_out + (int64_t)t * a.qo_token_stride + carried_off[j], carried[j]);
    } else if (TAIL && kind[j] == kTailK) {
      if (p.key_out) put(p.key_out + (int64_t)t * a.ko_token_stride + carried_off[j], carried[j]);
      if (ADDR != kNoCache && slot >= 0) put_cache(p.key_cache + slot + carried_off[j], carried[j]);
    }
  }
}

__host__ __device__ __forceinline__ RopeLayer only_layer(const RopeArgs& a) {
  return RopeLayer{a.query, a.key, a.value, a.query_out, a.key_out, a.key_cache, a.value_cache};
}
template <typename T, Addressing ADDR, int NTL>
__global__ __launch_bounds__(kThreads) void rope_pairs_kernel(typename LeanOf<ADDR>::type l) {
  const RopeArgs a = from_lean<T, ADDR, kPairs>(l);
  rope_pairs_lane<T, ADDR, NTL>(a, only_layer(a));
}
template <typename T, Addressing ADDR, int NTL>
__global__ __launch_bounds__(kThreads) void rope_rows_kernel(typename LeanOf<ADDR>::type l) {
  const RopeArgs a = from_lean<T, ADDR, kRows>(l);
  rope_rows_lane<T, ADDR, true, NTL>(a, only_layer(a));
}
template <typename T, Addressing ADDR, bool TAIL>
__global__ __launch_bounds__(kThreads) void rope_owner_kernel(typename LeanOf<ADDR>::type l) {
  const RopeArgs a = from_lean<T, ADDR, TAIL ? kOwnerTail : kOwner>(l);
  rope_owner_lane<T, ADDR, true, TAIL>(a, only_layer(a));
}
// Other index types, block sizes, and sizes that RopeLean does not hold; pairs: those sizes, and large page-table launches
template <typename T, Addressing ADDR, int NTL>
__global__ __launch_bounds__(kThreads) void rope_pairs_general_kernel(RopeArgs a) {
  rope_pairs_lane<T, ADDR, NTL>(a, only_layer(a));
}
template <typename T, Addressing ADDR, int NTL>
__global__ __launch_bounds__(kThreads) void rope_rows_general_kernel(RopeArgs a) {
  rope_rows_lane<T, ADDR, false, NTL>(a, only_layer(a));
}
template <typename T, Addressing ADDR>
__global__ __launch_bounds__(kThreads) void rope_owner_general_kernel(RopeArgs a) {
  rope_owner_lane<T, ADDR, false, true>(a, only_layer(a));
}

// The same for several layers of one step, blockIdx.z the layer, their pointers in the
// kernel arguments. A recorded step has every layer's buffers at hand before it begins;
// as one node per layer it is bound by what a node costs, not by its bytes. (A model loop
// has a layer's projections only after the layer before it, and records a launch per
// layer.) A replay with the index build, every layer's buffers its own, per layer -> one
// launch (us): 64 tokens x 28 + 4 heads x 128 x 28 layers 66.5 -> 18.1 (the index build
// alone 17.8), 256 x 32 + 8 heads x 32 109 -> 40, 717 tokens of those 199 -> 104, 3001 x
// 8 + 1 heads x 80 490 -> 257 (5.15 TB/s).
// A layer's value planes lie as far behind its key planes as every other layer's, so that 4 KiB, what a launch's
// arguments may take, name 82 layers.
constexpr int kLayersPerLaunch = 82;
struct RopeLayersArgs {
  RopeLean l;
  int64_t key_to_value;  // bytes
  struct {
    const char *query, *key, *value;
    char *query_out, *key_out, *key_cache;
  } layer[kLayersPerLaunch];
};
static_assert(sizeof(RopeLayersArgs) <= 4096, "kernel arguments");

template <typename T, VectorForm FORM, int NTL = 0>
__global__ __launch_bounds__(kThreads) void rope_layers_kernel(RopeLayersArgs args) {
  const auto& y = args.layer[blockIdx.z];
  const RopeLayer p{y.query, y.key, y.value, y.query_out, y.key_out, y.key_cache, y.key_cache + args.key_to_value};
  const RopeArgs a = from_lean<T, kSlots, FORM>(args.l);
  if constexpr (FORM == kPairs) rope_pairs_lane<T, kSlots, NTL>(a, p);
  else if constexpr (FORM == kRows) rope_rows_lane<T, kSlots, true, 0>(a, p);
  else rope_owner_lane<T, kSlots, true, FORM == kOwnerTail>(a, p);
}

// Element path: rows that are no whole number of aligned 16-byte vectors. One
// rotation pair or one pass-through element per lane, in this order: pairs of the
// Q heads then the K heads, elements beyond rotary_dim, V.
// Bound: instructions and 2- or 4-byte accesses at prefill sizes, the chain of
// dependent loads at decode sizes. So the rows are asked for first, the position's
// and the slot's chains run behind them, and the lean index forms are as above. us a
// launch with the row of cos/sin in LDS (first form), the slot's chain ahead of
// the rows, and now: 256 tokens x 15 heads x 36 in fp32 3.77, 5.26, 3.23; 256 x 40 x
// 128 in bf16 8.03, 7.14, 6.42; 2048 of those 40.4, 37.1, 30.0; 2048 x 32 x 80 with 20
// lanes rotated 33.9, 29.9, 23.3. 64 and 256 lanes to a workgroup are within 8 % of
// 128, more often slower.
template <typename T, Addressing ADDR, bool FAST>
__global__ __launch_bounds__(kThreads) void rope_element_kernel(RopeArgs a) {
  using VT = Vec<T>;
  constexpr int E = T::kBytes;
  const uint32_t t = blockIdx.x / a.groups_per_token;
  const uint32_t item = (blockIdx.x - t * a.groups_per_token) * a.threads + threadIdx.x;
  const int64_t pos = FAST ? (int64_t) reinterpret_cast<const int32_t*>(a.positions)[t] : index_of(a.positions, a.pos_bytes, t);
  const uint32_t rd = a.rotary_dim, half = rd >> 1, D = a.head_dim;
  const uint32_t heads = a.num_heads + a.num_kv_heads;
  const uint32_t rot_items = heads * half, tail_per_head = D - rd, head_items = rot_items + heads * tail_per_head;
  const bool pair = item < rot_items;
  const bool is_v = item >= head_items;
  if (is_v && (ADDR == kNoCache || item >= head_items + a.num_kv_heads * D)) return;
  const uint32_t i = pair ? item : item - rot_items;
  const uint32_t h = is_v ? 0 : pair ? i / half : i / tail_per_head;
  const uint32_t e = pair ? i - h * half : rd + (i - h * tail_per_head);
  const bool is_k = h >= a.num_heads;
  const int64_t off = is_v ? (int64_t)(item - head_items) * E : ((int64_t)(is_k ? h - a.num_heads : h) * D + e) * E;
  const char* in = (is_v ? a.value + (int64_t)t * a.v_token_stride
                         : is_k ? a.key + (int64_t)t * a.k_token_stride : a.query + (int64_t)t * a.q_token_stride) + off;
  const auto at = [](const char* p) { return *reinterpret_cast<const typename VT::Word*>(p); };
  const typename VT::Word x = at(in), y = pair ? at(in + (int64_t)half * E) : 0;
  if (pos < 0 || pos >= a.max_position) return;  // no cos/sin row: the token is left alone
  typename VT::Word cos_x = 0, cos_y = 0, sin_x = 0, sin_y = 0;
  if (pair) {
    const char* cs = a.cos_sin_cache + pos * (int64_t)(2 * rd) * E + (int64_t)e * E;
    cos_x = at(cs);
    cos_y = at(cs + (int64_t)half * E);
    sin_x = at(cs + (int64_t)rd * E);
    sin_y = at(cs + (int64_t)(rd + half) * E);
  }
  const int64_t slot = slot_offset<ADDR, FAST>(a, t, pos);
  typename VT::Word ox = x, oy = 0;
  if (pair) {  // narrowed once, the products contracted by hand: the same bits in every instantiation
    ox = VT::narrow(__builtin_fmaf(VT::wide(x), VT::wide(cos_x), -(VT::wide(y) * VT::wide(sin_x))));
    oy = VT::narrow(__builtin_fmaf(VT::wide(y), VT::wide(cos_y), VT::wide(x) * VT::wide(sin_y)));
  }
  const auto put = [](char* p, typename VT::Word w) { *reinterpret_cast<typename VT::Word*>(p) = w; };
  char* row = is_v ? nullptr : is_k ? a.key_out : a.query_out;
  if (row) {
    row += (int64_t)t * (is_k ? a.ko_token_stride : a.qo_token_stride) + off;
    put(row, ox);
    if (pair) put(row + (int64_t)half * E, oy);
  }
  if (ADDR != kNoCache && slot >= 0 && (is_v || is_k)) {
    char* out = (is_v ? a.value_cache : a.key_cache) + slot + off;
    put(out, ox);
    if (pair) put(out + (int64_t)half * E, oy);
  }
}

// Index types and block size that the lean instantiations take
template <Addressing ADDR>
bool fast_index(const RopeArgs& a) {
  return a.pos_bytes == 4 && (ADDR == kNoCache || a.bs_shift >= 0) && (ADDR != kSlots || a.slot_bytes == 8);
}

template <typename T, Addressing ADDR>
void launch_element(const RopeArgs& a, dim3 grid, dim3 block, hipStream_t s) {
  if (fast_index<ADDR>(a)) kvc::launch((rope_element_kernel<T, ADDR, true>), grid, block, 0, s, a);
  else kvc::launch((rope_element_kernel<T, ADDR, false>), grid, block, 0, s, a);
}

// Does a call's geometry fit the lean arguments?
bool lean_fits(const RopeArgs& a, int64_t E) {
  const auto u32 = [](int64_t v) { return v >= 0 && v <= (int64_t)UINT32_MAX; };
  const bool strides = u32(a.q_token_stride) && u32(a.k_token_stride) && u32(a.v_token_stride) && u32(a.qo_token_stride) &&
                       u32(a.ko_token_stride) && a.head_dim * E / 16 <= UINT8_MAX;
  const bool cache = !a.key_cache || (u32(a.cache_block_stride) && u32(a.cache_slot_stride) && u32(a.num_cache_blocks));
  return strides && cache && a.num_heads <= UINT16_MAX && a.num_kv_heads <= UINT16_MAX;
}

// Counts that 32-bit indices are compared with: beyond every such index they are all the same
uint32_t beyond_int32(int64_t n) { return (uint32_t)std::min<int64_t>(n, int64_t(1) << 31); }

template <Addressing ADDR>
typename LeanOf<ADDR>::type lean_of(const RopeArgs& a, int64_t E) {
  typename LeanOf<ADDR>::type l{};
  l.query = a.query; l.key = a.key; l.value = a.value;
  l.query_out = a.query_out; l.key_out = a.key_out; l.key_cache = a.key_cache; l.value_cache = a.value_cache;
  l.positions = a.positions; l.cos_sin_cache = a.cos_sin_cache; l.slot_mapping = a.slot_mapping;
  l.q_token_stride = (uint32_t)a.q_token_stride; l.k_token_stride = (uint32_t)a.k_token_stride;
  l.v_token_stride = (uint32_t)a.v_token_stride;
  l.qo_token_stride = (uint32_t)a.qo_token_stride; l.ko_token_stride = (uint32_t)a.ko_token_stride;
  l.max_position = beyond_int32(a.max_position);
  l.cache_block_stride = (uint32_t)a.cache_block_stride; l.cache_slot_stride = (uint32_t)a.cache_slot_stride;
  l.num_cache_blocks = (uint32_t)a.num_cache_blocks;
  l.split_magic = a.split_magic;
  l.num_heads = (uint16_t)a.num_heads; l.num_kv_heads = (uint16_t)a.num_kv_heads;
  l.pairs_per_head = (uint8_t)a.pairs_per_head; l.vecs_per_head = (uint8_t)(a.head_dim * E / 16);
  l.bs_shift = (uint8_t)std::max(a.bs_shift, 0);
  l.shape = (uint8_t)(a.threads / 64 * 2 + (a.cache_nt ? 1 : 0));
  if constexpr (ADDR == kPages) {
    l.batch_indices = a.batch_indices; l.kv_indices = a.kv_indices; l.kv_indptr = a.kv_indptr;
    l.batch_size = beyond_int32(a.batch_size); l.num_kv_indices = beyond_int32(a.num_kv_indices);
  }
  return l;
}

template <typename T, Addressing ADDR, int NTL>
void launch_vector(const RopeArgs& a, VectorForm form, bool lean, dim3 grid, dim3 block, hipStream_t s) {
  // By page table what RopeLeanPages folds away stands ahead of three steps of loads. Up to 4 MiB of rows the host's share
  // of a launch is the longer one; beyond, the device's (us, RopeArgs and this: 700 tokens x 32 + 8 heads x 128 4.2 and 4.4,
  // 256 x 64 + 8 in fp32 4.8 and 5.2, 1500 x 32 + 8 x 64 4.3 and 4.5; 1 % over all sizes).
  const bool large = ADDR == kPages && (int64_t)grid.y * (a.num_heads + 2 * a.num_kv_heads) * a.head_dim * T::kBytes > (4 << 20);
  if (form == kPairs && (!lean || large)) kvc::launch((rope_pairs_general_kernel<T, ADDR, NTL>), grid, block, 0, s, a);
  else if (form == kPairs) kvc::launch((rope_pairs_kernel<T, ADDR, NTL>), grid, block, 0, s, lean_of<ADDR>(a, T::kBytes));
  else if (lean) kvc::launch((rope_rows_kernel<T, ADDR, NTL>), grid, block, 0, s, lean_of<ADDR>(a, T::kBytes));
  else kvc::launch((rope_rows_general_kernel<T, ADDR, NTL>), grid, block, 0, s, a);
}

template <typename T, Addressing ADDR>
void launch_vector(const RopeArgs& a, VectorForm form, int ntl, dim3 grid, dim3 block, hipStream_t s) {
  const bool lean = fast_index<ADDR>(a) && lean_fits(a, T::kBytes);
  if (form == kOwner || form == kOwnerTail) {
    if (!lean) kvc::launch((rope_owner_general_kernel<T, ADDR>), grid, block, 0, s, a);
    else if (form == kOwner) kvc::launch((rope_owner_kernel<T, ADDR, false>), grid, block, 0, s, lean_of<ADDR>(a, T::kBytes));
    else kvc::launch((rope_owner_kernel<T, ADDR, true>), grid, block, 0, s, lean_of<ADDR>(a, T::kBytes));
    return;
  }
  switch (ntl) {
    case 0: launch_vector<T, ADDR, 0>(a, form, lean, grid, block, s); break;
    case 1: launch_vector<T, ADDR, 1>(a, form, lean, grid, block, s); break;
    case 2: launch_vector<T, ADDR, 2>(a, form, lean, grid, block, s); break;
    default: launch_vector<T, ADDR, 3>(a, form, lean, grid, block, s); break;
  }
}

template <typename T>
int launch_rope(RopeArgs a, int64_t num_tokens, VectorForm form, int ntl, unsigned threads, hipStream_t s) {
  if (form == kElements) {
    const dim3 grid((unsigned)(num_tokens * a.groups_per_token)), block(threads);
    if (!a.key_cache) launch_element<T, kNoCache>(a, grid, block, s);
    else if (a.batch_indices) launch_element<T, kPages>(a, grid, block, s);
    else launch_element<T, kSlots>(a, grid, block, s);
    KVC_HIP(hipGetLastError());
    kvc::record_rotation(T::kBytes, form, (int)threads, grid.x, 0);
    return KVC_OK;
  }
  constexpr int64_t kMaxY = 65535;  // tokens of one launch
  const int64_t slot_step = a.slot_bytes, pos_step = a.pos_bytes;
  for (int64_t t0 = 0; t0 < num_tokens; t0 += kMaxY) {
    const dim3 grid(a.groups_per_token, (unsigned)std::min(kMaxY, num_tokens - t0)), block(threads);
    if (!a.key_cache) launch_vector<T, kNoCache>(a, form, ntl, grid, block, s);
    else if (a.batch_indices) launch_vector<T, kPages>(a, form, ntl, grid, block, s);
    else launch_vector<T, kSlots>(a, form, ntl, grid, block, s);
    KVC_HIP(hipGetLastError());
    kvc::record_rotation(16, form, (int)threads, (int64_t)grid.x * grid.y,
                         form == kOwner || form == kOwnerTail ? 0 : ntl);
    a.query += kMaxY * a.q_token_stride;
    a.key += kMaxY * a.k_token_stride;
    if (a.value) a.value += kMaxY * a.v_token_stride;
    a.query_out += kMaxY * a.qo_token_stride;
    if (a.key_out) a.key_out += kMaxY * a.ko_token_stride;
    a.positions = (const char*)a.positions + kMaxY * pos_step;
    if (a.slot_mapping) a.slot_mapping = (const char*)a.slot_mapping + kMaxY * slot_step;
    if (a.batch_indices) a.batch_indices += kMaxY;
  }
  return KVC_OK;
}

// Several layers of slot-mapped writes, as many to a launch as the arguments hold
template <typename T>
int launch_rope_layers(RopeArgs a, const RopeLayer* layers, int64_t num_layers, int64_t num_tokens, VectorForm form,
                       bool nt, unsigned threads, hipStream_t s) {
  RopeLayersArgs args{};
  for (int64_t l0 = 0; l0 < num_layers; l0 += kLayersPerLaunch) {
    const int64_t n = std::min<int64_t>(kLayersPerLaunch, num_layers - l0);
    args.l = lean_of<kSlots>(a, T::kBytes);
    args.key_to_value = a.value_cache - a.key_cache;
    for (int64_t l = 0; l < n; ++l) {
      const RopeLayer& p = layers[l0 + l];
      args.layer[l] = {p.query, p.key, p.value, p.query_out, p.key_out, p.key_cache};
    }
    const dim3 grid(a.groups_per_token, (unsigned)num_tokens, (unsigned)n), block(threads);
    if (form == kPairs && nt) kvc::launch((rope_layers_kernel<T, kPairs, 3>), grid, block, 0, s, args);
    else if (form == kPairs) kvc::launch((rope_layers_kernel<T, kPairs>), grid, block, 0, s, args);
    else if (form == kRows) kvc::launch((rope_layers_kernel<T, kRows>), grid, block, 0, s, args);
    else if (form == kOwner) kvc::launch((rope_layers_kernel<T, kOwner>), grid, block, 0, s, args);
    else kvc::launch((rope_layers_kernel<T, kOwnerTail>), grid, block, 0, s, args);
    KVC_HIP(hipGetLastError());
    kvc::record_rotation(16, form, (int)threads, (int64_t)grid.x * grid.y * grid.z, form == kPairs && nt ? 3 : 0);
  }
  return KVC_OK;
}

struct RopeGeom {
  int64_t num_tokens, num_heads, num_kv_heads, head_dim, rotary_dim, max_position;
  int64_t q_token_stride, k_token_stride, v_token_stride, qo_token_stride, ko_token_stride;  // elements
  int dtype;
};

struct CacheGeom {
  void* key_cache;
  void* value_cache;
  const void* slot_mapping;
  int slot_bytes;
  const int32_t* batch_indices;
  const int32_t* kv_indices;
  const int32_t* kv_indptr;
  int64_t batch_size, num_kv_indices;
  int64_t block_size, cache_block_stride, cache_slot_stride, num_cache_blocks;  // strides in elements
};

// Does a byte range that one layer writes meet anything that another layer reads or writes?
// Then the layers depend on their order, and one launch has none. Bytes: of the rows and of a
// layer's whole cache.
struct LayerExtents {
  int64_t query, key, value, query_out, key_out, cache;
};
bool layers_depend(const RopeLayer* layers, int64_t n, const LayerExtents& e) {
  struct Range {
    const char *begin, *end;
  };
  const auto range = [](const char* p, int64_t bytes) { return Range{p, p ? p + bytes : p}; };
  for (int64_t i = 0; i < n; ++i) {
    const RopeLayer& w = layers[i];
    for (int64_t j = 0; j < n; ++j) {
      if (j == i) continue;
      const RopeLayer& o = layers[j];
      for (const Range& x : {range(w.query_out, e.query_out), range(w.key_out, e.key_out), range(w.key_cache, e.cache)})
        for (const Range& y : {range(o.query, e.query), range(o.key, e.key), range(o.value, e.value),
                               range(o.query_out, e.query_out), range(o.key_out, e.key_out), range(o.key_cache, e.cache)})
          if (x.begin < y.end && y.begin < x.end) return true;
    }
  }
  return false;
}

// Layers whose rows are not those of a layer before
int64_t distinct_rows(const RopeLayer* layers, int64_t n) {
  int64_t distinct = 0;
  for (int64_t i = 0; i < n; ++i) {
    int64_t j = 0;
    while (j < i && layers[j].query != layers[i].query) ++j;
    distinct += j == i;
  }
  return distinct;
}

// Does a row that a layer writes meet a Q or K row that it reads? (V passes through, vector by vector.) Bytes.
bool writes_its_input(const RopeLayer& p, const RopeGeom& g, const CacheGeom* c, int64_t E) {
  typedef __int128 Wide;  // a cache may be said to have any number of blocks
  const auto rows = [&](int64_t stride, int64_t row) { return ((Wide)(g.num_tokens - 1) * stride + row) * E; };
  const auto meet = [](const char* x, Wide x_bytes, const char* y, Wide y_bytes) {
    const Wide bx = (uintptr_t)x, by = (uintptr_t)y;
    return x && bx < by + y_bytes && by < bx + x_bytes;
  };
  const int64_t q_row = g.num_heads * g.head_dim, k_row = g.num_kv_heads * g.head_dim;
  const auto meets_input = [&](const char* out, Wide bytes) {
    return meet(out, bytes, p.query, rows(g.q_token_stride, q_row)) || meet(out, bytes, p.key, rows(g.k_token_stride, k_row));
  };
  return meets_input(p.query_out, rows(g.qo_token_stride, q_row)) ||
         meets_input(p.key_out, rows(g.ko_token_stride, k_row)) ||
         (c && c->num_cache_blocks > 0 &&
          meets_input(p.key_cache, ((Wide)(c->num_cache_blocks - 1) * c->cache_block_stride +
                                    (Wide)(c->block_size - 1) * c->cache_slot_stride + k_row) * E));
}

constexpr int kLayerByLayer = 1;  // run_rope: nothing launched, the layers' buffers do not suit one launch

// With `layers` (the first of them the buffers named before) every layer goes into one launch, or none does.
int run_rope(const char* fn, const void* query, const void* key, const void* value,
             void* query_out, void* key_out, const void* positions, int pos_bytes,
             const void* cos_sin_cache, const RopeGeom& g, const CacheGeom* c, void* stream,
             const RopeLayer* layers = nullptr, int64_t num_layers = 0) {
  int E;
  switch (g.dtype) {
    case KVC_DTYPE_BF16: case KVC_DTYPE_F16: E = 2; break;
    case KVC_DTYPE_F32: E = 4; break;
    default: return fail(KVC_ERR_UNSUPPORTED, "%s: dtype %d (need bf16, f16 or f32)", fn, g.dtype);
  }
  if (g.num_tokens < 0 || g.num_heads < 0 || g.num_kv_heads < 0 || g.head_dim <= 0 ||
      g.rotary_dim < 0 || g.max_position < 0)
    return fail(KVC_ERR_INVALID_ARG, "%s: negative size", fn);
  if (g.rotary_dim > g.head_dim || (g.rotary_dim & 1))
    return fail(KVC_ERR_INVALID_ARG, "%s: rotary_dim %lld must be even and <= head_dim %lld", fn,
                (long long)g.rotary_dim, (long long)g.head_dim);
  if (g.rotary_dim > kMaxRotaryDim)
    return fail(KVC_ERR_UNSUPPORTED, "%s: rotary_dim %lld exceeds %d", fn, (long long)g.rotary_dim,
                kMaxRotaryDim);
  if (pos_bytes != 4 && pos_bytes != 8)
    return fail(KVC_ERR_UNSUPPORTED, "%s: pos_bytes=%d (need 4 or 8)", fn, pos_bytes);
  if (g.num_tokens > 0x7fffffffll || g.num_heads + g.num_kv_heads > 0xffffll)
    return fail(KVC_ERR_UNSUPPORTED, "%s: too many tokens or heads", fn);
  if (g.num_tokens == 0 || g.num_heads + g.num_kv_heads == 0) return KVC_OK;
  if (!query || !key || !query_out || !positions || !cos_sin_cache)
    return fail(KVC_ERR_INVALID_ARG, "%s: null pointer", fn);
  if (!c && !key_out) return fail(KVC_ERR_INVALID_ARG, "%s: no destination for the rotated key", fn);
  if (g.q_token_stride < g.num_heads * g.head_dim || g.qo_token_stride < g.num_heads * g.head_dim ||
      g.k_token_stride < g.num_kv_heads * g.head_dim ||
      (key_out && g.ko_token_stride < g.num_kv_heads * g.head_dim))
    return fail(KVC_ERR_INVALID_ARG, "%s: token stride smaller than a row", fn);

  RopeArgs a{};
  a.query = (const char*)query;
  a.key = (const char*)key;
  a.value = (const char*)value;
  a.query_out = (char*)query_out;
  a.key_out = (char*)key_out;
  a.positions = positions;
  a.pos_bytes = pos_bytes;
  a.cos_sin_cache = (const char*)cos_sin_cache;
  a.max_position = g.max_position;
  a.num_heads = (uint32_t)g.num_heads;
  a.num_kv_heads = (uint32_t)g.num_kv_heads;
  a.head_dim = (uint32_t)g.head_dim;
  a.rotary_dim = (uint32_t)g.rotary_dim;
  a.q_token_stride = g.q_token_stride * E;
  a.k_token_stride = g.k_token_stride * E;
  a.v_token_stride = g.v_token_stride * E;
  a.qo_token_stride = g.qo_token_stride * E;
  a.ko_token_stride = g.ko_token_stride * E;

  uint64_t in_align = (uintptr_t)query | (uintptr_t)key | (uint64_t)a.q_token_stride | (uint64_t)a.k_token_stride;
  uint64_t out_align = (uintptr_t)query_out | (uintptr_t)key_out | (uint64_t)a.qo_token_stride | (uint64_t)a.ko_token_stride;
  if (c) {
    if (!value || !c->key_cache || !c->value_cache)
      return fail(KVC_ERR_INVALID_ARG, "%s: null value/cache pointer", fn);
    if (g.v_token_stride < g.num_kv_heads * g.head_dim)
      return fail(KVC_ERR_INVALID_ARG, "%s: value token stride smaller than a row", fn);
    if (c->block_size <= 0 || c->num_cache_blocks < 0 || c->cache_block_stride < 0 ||
        c->cache_slot_stride < g.num_kv_heads * g.head_dim)
      return fail(KVC_ERR_INVALID_ARG, "%s: bad cache geometry", fn);
    if (c->batch_indices) {
      if (!c->kv_indices || !c->kv_indptr || c->batch_size < 0 || c->num_kv_indices < 0)
        return fail(KVC_ERR_INVALID_ARG, "%s: bad page-table arguments", fn);
      if (pos_bytes != 4)
        return fail(KVC_ERR_UNSUPPORTED, "%s: page-table addressing takes int32 positions", fn);
    } else {
      if (!c->slot_mapping) return fail(KVC_ERR_INVALID_ARG, "%s: null slot_mapping", fn);
      if (c->slot_bytes != 4 && c->slot_bytes != 8)
        return fail(KVC_ERR_UNSUPPORTED, "%s: slot_bytes=%d (need 4 or 8)", fn, c->slot_bytes);
    }
    a.key_cache = (char*)c->key_cache;
    a.value_cache = (char*)c->value_cache;
    a.slot_mapping = c->slot_mapping;
    a.slot_bytes = c->slot_bytes;
    a.batch_indices = c->batch_indices;
    a.kv_indices = c->kv_indices;
    a.kv_indptr = c->kv_indptr;
    a.batch_size = c->batch_size;
    a.num_kv_indices = c->num_kv_indices;
    a.block_size = c->block_size;
    a.bs_shift = log2_exact(c->block_size);
    a.cache_block_stride = c->cache_block_stride * E;
    a.cache_slot_stride = c->cache_slot_stride * E;
    a.num_cache_blocks = c->num_cache_blocks;
    in_align |= (uintptr_t)value | (uint64_t)a.v_token_stride;
    out_align |= (uintptr_t)c->key_cache | (uintptr_t)c->value_cache | (uint64_t)a.cache_block_stride |
                 (uint64_t)a.cache_slot_stride;
  }
  bool in_place = writes_its_input(only_layer(a), g, c, E);
  for (int64_t l = 0; l < num_layers; ++l) {
    const RopeLayer& p = layers[l];
    in_place = in_place || writes_its_input(p, g, c, E);
    in_align |= (uintptr_t)p.query | (uintptr_t)p.key | (uintptr_t)p.value;
    out_align |= (uintptr_t)p.query_out | (uintptr_t)p.key_out | (uintptr_t)p.key_cache | (uintptr_t)p.value_cache;
  }
  // 16-byte vectors need aligned rows and halves that hold whole vectors (and offsets inside a row that fit
  // 32 bits); the cos/sin table may start anywhere
  const int ev = 16 / E;
  const int64_t heads = g.num_heads + g.num_kv_heads;
  const bool vector = (in_align | out_align) % 16 == 0 && heads * g.head_dim * E <= (int64_t(1) << 29) &&
                      (g.rotary_dim / 2) % ev == 0 && (g.head_dim - g.rotary_dim) % ev == 0 && g.head_dim % ev == 0;
  int ntl = kvc::g_rope_tune.nt & 3;
  VectorForm form = kElements;
  unsigned threads = (unsigned)kvc::g_rope_tune.threads;
  const bool fixed = threads == 64 || threads == 128 || threads == 192 || threads == 256;
  if (vector) {
    const int64_t half = (g.rotary_dim / 2) * E, v_items = c ? g.num_kv_heads * g.head_dim / ev : 0;
    const bool fast = !c ? fast_index<kNoCache>(a) : a.batch_indices ? fast_index<kPages>(a) : fast_index<kSlots>(a);
    a.v_items = (uint32_t)v_items;
    a.cache_nt = g.num_tokens * v_items * 32 > (int64_t(3) << 20);
    a.pairs_per_head = (uint32_t)((g.rotary_dim / 2) / ev);
    const int64_t pair_lanes = heads * a.pairs_per_head, extras = v_items + heads * ((g.head_dim - g.rotary_dim) / ev);
    const int64_t bytes = g.num_tokens * heads * g.head_dim * E * std::max<int64_t>(num_layers, 1);  // Q and K rows
    // Whole heads, as the pair and the owner form without tails take them
    const bool whole = fast && g.rotary_dim == g.head_dim && v_items <= pair_lanes;
    const bool lines = half % 64 == 0 && out_align % 64 == 0;
    // Small launches are latency, and the owner form has the shortest chain (launches of a recorded step of 32 layers
    // alone, then with a gather of the new cache rows behind each, us; owner and pairs: 16 tokens x 28 + 4 heads x 128
    // 2.23 and 2.28, 3.83 and 4.14; 64 of those (512 KiB) 2.29 and 2.31, 3.89 and 4.17; 192 2.46 and 2.42, 4.45 and 4.33;
    // with wider cache rows the pair form's reader makes up for it: 16 x 32 + 8 x 128 2.19 and 2.22, 4.15 and 4.10.
    // Owner and rows: 64 tokens x 28 + 4 x 96 2.26 and 2.51, 3.88 and 4.42; 192 x 32 + 8 x 96 (1.4 MiB) 2.50 and 2.67,
    // 4.84 and 5.28; 400 x 32 + 8 x 80 (2.4 MiB) 2.90 and 2.84; in fp32, 400 lanes a token, 64 of those 2.67 and 2.39)
    const bool small = lines ? bytes <= (512 << 10) && g.num_kv_heads * g.head_dim * E < 1536
                             : bytes <= (2 << 20) && pair_lanes <= 320;
    // Large ones whose token is one workgroup as pairs and three, of which the last is mostly idle, as rows (32 + 8 heads
    // x 96 in bf16, owner and rows, us: 838 tokens, 6 MiB, 4.6 and 4.5, 1600 6.8 and 6.9, 2048 7.5 and 8.2, 5000 15.3 and
    // 16.9, 8192 27.3 and 27.3)
    const int64_t row_lanes = lanes_of<int64_t>(kRows, g.num_heads, g.num_kv_heads, a.pairs_per_head, g.head_dim / ev, c);
    const bool one_group = !lines && bytes >= (8 << 20) && pair_lanes <= kThreads && row_lanes > kThreads;
    // Halves of 64 bytes are whole pieces of half a line each; from 16 MiB of Q and K rows on, whole lines are worth
    // more than the pair form's fewer lanes (pairs and rows, us: 32 + 8 heads x 64 in bf16, 1024 tokens 3.57 and 3.73,
    // 4096 10.13 and 10.17, with a reader of query_out 16.08 and 15.84, 6000 13.3 and 13.3, 24.7 and 22.8, 8192 21.7
    // and 20.0, 31.1 and 29.0)
    const bool pairs = lines && !(half == 64 && g.num_tokens * heads * g.head_dim * E >= (int64_t(16) << 20));
    // In place the pair form stays, which reads no vector that another lane writes, and the owner form stands in for rows
    if (whole && (small || one_group)) form = kOwner;
    else if (whole && pairs) form = kPairs;
    else if (!in_place || !g.rotary_dim) form = kRows;
    else form = extras > v_items || v_items > pair_lanes ? kOwnerTail : kOwner;
    // From 40 MiB of Q, K and V rows on the pair form's loads are non-temporal. Beside what the launch writes and what ran
    // before it, the projection that wrote these rows first of all, the last-level cache no longer holds them well, and
    // plain loads push out dirty lines. us a launch, plain and non-temporal: the same rows again and again, unchanged; four sets
    // in turn; rows just written by a kernel in front (its time included); with a copy of query_out behind it as well.
    // The first is not how rows come, and loses from 64 MiB on:
    //   32 + 8 heads x 128, 30 MiB   9.9 11.6    11.1 12.5    21.8 21.9    28.9 28.8
    //     36 MiB                     12.9 13.0   13.5 14.1    25.2 25.4    33.1 33.4
    //     41 MiB                     14.8 14.1   16.9 15.6    28.2 28.2    36.9 37.0
    //     64 MiB                     22.0 22.9   25.7 23.2    41.8 42.0    57.6 56.0
    //     100 MiB                    33.3 34.8   38.1 35.8    65.6 65.8    96.0 88.1
    //   64 + 8, 41 MiB               14.5 14.1   17.0 15.7    28.0 28.3    38.8 38.9
    //     64 MiB                     21.7 21.0   25.8 22.7    41.5 41.9    62.5 58.4
    //     128 MiB                    41.3 45.8   47.9 45.8    89.3 84.4    145.6 125.5
    // Several layers in one launch: from 128 MiB of rows on that are not those of another layer as well (us a launch, plain and
    // non-temporal; all layers' rows their own, 28 x 28 + 4 heads x 128: 24 MiB 8.9 11.6, 64 15.2 15.7, 128 42.2 42.3, 200
    // 75.3 62.5, 400 149 139, 800 300 283; 32 x 32 + 8: 128 43.3 42.0, 260 96.8 80.6, 800 290 276; four sets of rows
    // that the layers take in turn: 28 x 7.1 MiB 45.6 62.0, 28 x 28.6 284 286, 28 x 57 603 580, 80 x 20 478 584).
    // Steps of the rows form lose by it (8192 tokens x 24 layers, 32 + 8 heads x 80, 32 rotated, 570 and 587 us; 16 layers
    // of 32 + 8 x 64 323 and 330), and so does a rotation without the cache (5000 x 32 + 8 x 128, 32 layers, 954 and 961).
    const int64_t layer_bytes = g.num_tokens * (heads + g.num_kv_heads) * g.head_dim * E;
    if (!kvc::g_rope_tune.nt && form == kPairs && c &&
        (layers ? layer_bytes * distinct_rows(layers, num_layers) >= (int64_t(128) << 20) : layer_bytes >= (int64_t(40) << 20)))
      ntl = 3;
    if (form != kRows) {
      a.split = a.pairs_per_head;
      a.lanes_per_token = (uint32_t)lanes_of<int64_t>(form, g.num_heads, g.num_kv_heads, a.pairs_per_head, g.head_dim / ev, c);
    } else {
      a.split = (uint32_t)(g.head_dim / ev);
      a.head_step = (uint32_t)((heads + (c ? g.num_kv_heads : 0) + 1) / 2);
      a.lanes_per_token = (uint32_t)row_lanes;
    }
    const int64_t lanes = a.lanes_per_token;
    // exact for every lane where lanes * split < 2^32 (pairs: lanes < 2^25, at most 64 pair-vectors per head)
    a.split_magic = a.split > 1 && lanes * a.split < (int64_t(1) << 32)
                        ? (uint32_t)(((uint64_t(1) << 32) + a.split - 1) / a.split) : 0;
    // The largest workgroup that cuts a token into an ODD number of workgroups. They are dealt round-robin to
    // the 8 XCDs; with an even number every second XCD gets only first halves (with the V vectors), the others
    // only the short last ones: 40 heads x 128 (5 wavefronts), 2048 tokens, as 3 x 128 lanes 9.5 us, as 5 x 64
    // 9.7, as 2 x 192 10.5, as 2 x 256 11.3; 40 heads x 64 (3 wavefronts) as 1 x 256 6.3, as 2 x 128 7.0.
    const int64_t waves = (lanes + 63) / 64;
    if (!fixed) {
      threads = 256;
      for (unsigned w = 4; w >= 1; --w)
        if ((waves + w - 1) / w % 2 == 1) {
          threads = 64 * w;
          break;
        }
    }
    a.groups_per_token = (uint32_t)std::max<int64_t>(1, (lanes + threads - 1) / threads);
  } else {
    const int64_t items = heads * (g.rotary_dim / 2) + heads * (g.head_dim - g.rotary_dim) +
                          (c ? g.num_kv_heads * g.head_dim : 0);
    if (!fixed) threads = 128;
    a.groups_per_token = (uint32_t)std::max<int64_t>(1, (items + threads - 1) / threads);
  }
  if (g.num_tokens * (int64_t)a.groups_per_token > 0x7fffffffll)
    return fail(KVC_ERR_UNSUPPORTED, "%s: launch of %lld workgroups is too large", fn,
                (long long)(g.num_tokens * (int64_t)a.groups_per_token));
  if (c && c->batch_indices && (c->batch_size == 0 || c->num_kv_indices == 0)) {  // the write skips every token
    a.key_cache = nullptr;
    a.v_items = 0;
  }
  a.threads = threads;
  hipStream_t s = (hipStream_t)stream;
  if (layers) {
    if (form == kElements || !c->slot_mapping || !lean_fits(a, E) || c->slot_bytes != 8 || pos_bytes != 4 || a.bs_shift < 0 ||
        (kvc::g_rope_tune.nt & 3) || g.num_tokens > 65535)
      return kLayerByLayer;
    switch (g.dtype) {
      case KVC_DTYPE_BF16: return launch_rope_layers<BF16>(a, layers, num_layers, g.num_tokens, form, ntl != 0, threads, s);
      case KVC_DTYPE_F16: return launch_rope_layers<F16>(a, layers, num_layers, g.num_tokens, form, ntl != 0, threads, s);
      default: return launch_rope_layers<F32>(a, layers, num_layers, g.num_tokens, form, ntl != 0, threads, s);
    }
  }
  switch (g.dtype) {
    case KVC_DTYPE_BF16: return launch_rope<BF16>(a, g.num_tokens, form, ntl, threads, s);
    case KVC_DTYPE_F16: return launch_rope<F16>(a, g.num_tokens, form, ntl, threads, s);
    default: return launch_rope<F32>(a, g.num_tokens, form, ntl, threads, s);
  }
}

}  // namespace

extern "C" {

int kvc_rotary_pos_emb(const void* query, const void* key, const void* positions, int pos_bytes,
                       const void* cos_sin_cache, int64_t max_position, int64_t num_tokens,
                       int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                       int64_t rotary_dim, int64_t q_token_stride, int64_t k_token_stride,
                       void* query_out, void* key_out, int64_t qo_token_stride,
                       int64_t ko_token_stride, int dtype, void* stream) {
  RopeGeom g{num_tokens, num_heads, num_kv_heads, head_dim, rotary_dim, max_position,
             q_token_stride, k_token_stride, 0, qo_token_stride, ko_token_stride, dtype};
  return run_rope("kvc_rotary_pos_emb", query, key, nullptr, query_out, key_out, positions,
                  pos_bytes, cos_sin_cache, g, nullptr, stream);
}

int kvc_rotary_pos_emb_and_cache(const void* query, const void* key, const void* value,
                                 const void* positions, int pos_bytes, const void* cos_sin_cache,
                                 int64_t max_position, int64_t num_tokens, int64_t num_heads,
                                 int64_t num_kv_heads, int64_t head_dim, int64_t rotary_dim,
                                 int64_t q_token_stride, int64_t k_token_stride,
                                 int64_t v_token_stride, void* query_out, void* key_out,
                                 int64_t qo_token_stride, int64_t ko_token_stride,
                                 void* key_cache, void* value_cache, const void* slot_mapping,
                                 int slot_bytes, int64_t block_size, int64_t cache_block_stride,
                                 int64_t cache_slot_stride, int64_t num_cache_blocks, int dtype,
                                 void* stream) {
  RopeGeom g{num_tokens, num_heads, num_kv_heads, head_dim, rotary_dim, max_position,
             q_token_stride, k_token_stride, v_token_stride, qo_token_stride, ko_token_stride, dtype};
  CacheGeom c{key_cache, value_cache, slot_mapping, slot_bytes, nullptr, nullptr, nullptr, 0, 0,
              block_size, cache_block_stride, cache_slot_stride, num_cache_blocks};
  return run_rope("kvc_rotary_pos_emb_and_cache", query, key, value, query_out, key_out, positions,
                  pos_bytes, cos_sin_cache, g, &c, stream);
}

int kvc_rotary_pos_emb_and_append_paged(const void* query, const void* key, const void* value,
                                        const int32_t* batch_indices, const int32_t* positions,
                                        const void* cos_sin_cache, int64_t max_position,
                                        int64_t nnz, int64_t num_heads, int64_t num_kv_heads,
                                        int64_t head_dim, int64_t rotary_dim,
                                        int64_t q_token_stride, int64_t k_token_stride,
                                        int64_t v_token_stride, void* query_out, void* key_out,
                                        int64_t qo_token_stride, int64_t ko_token_stride,
                                        void* paged_kv_cache, const int32_t* kv_indices,
                                        const int32_t* kv_indptr, int64_t batch_size,
                                        int64_t num_kv_indices, int64_t page_size,
                                        int64_t page_stride, int64_t num_pages, int dtype,
                                        void* stream) {
  if (nnz > 0 && !batch_indices)
    return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_pos_emb_and_append_paged: null batch_indices");
  if (num_kv_heads < 0 || head_dim <= 0 || page_size <= 0)
    return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_pos_emb_and_append_paged: bad H/D/page_size");
  const int64_t row = num_kv_heads * head_dim;
  if (page_stride < 2 * page_size * row)
    return fail(KVC_ERR_INVALID_ARG,
                "kvc_rotary_pos_emb_and_append_paged: page_stride %lld < 2*page_size*H*D",
                (long long)page_stride);
  const int E = dtype == KVC_DTYPE_F32 ? 4 : 2;
  RopeGeom g{nnz, num_heads, num_kv_heads, head_dim, rotary_dim, max_position,
             q_token_stride, k_token_stride, v_token_stride, qo_token_stride, ko_token_stride, dtype};
  char* vc = paged_kv_cache ? (char*)paged_kv_cache + page_size * row * E : nullptr;
  CacheGeom c{paged_kv_cache, vc, nullptr, 0, batch_indices, kv_indices, kv_indptr, batch_size,
              num_kv_indices, page_size, page_stride, row, num_pages};
  return run_rope("kvc_rotary_pos_emb_and_append_paged", query, key, value, query_out, key_out,
                  positions, 4, cos_sin_cache, g, &c, stream);
}

// ---- per-step plan of the fused rotation + page-table write ------------------
struct kvc_rotary_plan {
  const int32_t* batch_indices;
  const int32_t* positions;
  const void* cos_sin_cache;
  const int32_t* kv_indices;
  const int32_t* kv_indptr;
  int64_t max_position, nnz, num_heads, num_kv_heads, head_dim, rotary_dim;
  int64_t batch_size, num_kv_indices, page_size;
  int dtype;
  const int64_t* slots;  // resolved by kvc_rotary_plan_resolve_slots, else null
};

int kvc_rotary_plan_create(const int32_t* batch_indices, const int32_t* positions,
                           const void* cos_sin_cache, int64_t max_position, int64_t nnz,
                           int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                           int64_t rotary_dim, const int32_t* kv_indices,
                           const int32_t* kv_indptr, int64_t batch_size, int64_t num_kv_indices,
                           int64_t page_size, int dtype, kvc_rotary_plan** out) {
  if (!out) return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_create: null out");
  *out = nullptr;
  if (dtype != KVC_DTYPE_BF16 && dtype != KVC_DTYPE_F16 && dtype != KVC_DTYPE_F32)
    return fail(KVC_ERR_UNSUPPORTED, "kvc_rotary_plan_create: dtype %d (need bf16, f16 or f32)", dtype);
  if (nnz < 0 || num_heads < 0 || num_kv_heads < 0 || head_dim <= 0 || rotary_dim < 0 ||
      max_position < 0 || batch_size < 0 || num_kv_indices < 0 || page_size <= 0)
    return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_create: bad size");
  if (rotary_dim > head_dim || (rotary_dim & 1))
    return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_create: rotary_dim %lld must be even and <= head_dim %lld",
                (long long)rotary_dim, (long long)head_dim);
  if (rotary_dim > kMaxRotaryDim)
    return fail(KVC_ERR_UNSUPPORTED, "kvc_rotary_plan_create: rotary_dim %lld exceeds %d",
                (long long)rotary_dim, kMaxRotaryDim);
  if (nnz > 0 && (!batch_indices || !positions || !cos_sin_cache || !kv_indices || !kv_indptr))
    return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_create: null pointer");
  kvc_rotary_plan* p = new (std::nothrow) kvc_rotary_plan{
      batch_indices, positions, cos_sin_cache, kv_indices, kv_indptr, max_position, nnz, num_heads,
      num_kv_heads, head_dim, rotary_dim, batch_size, num_kv_indices, page_size, dtype, nullptr};
  if (!p) return fail(KVC_ERR_HIP, "kvc_rotary_plan_create: out of host memory");
  *out = p;
  return KVC_OK;
}

int kvc_rotary_plan_run(const kvc_rotary_plan* plan, const void* query, const void* key,
                        const void* value, int64_t q_token_stride, int64_t k_token_stride,
                        int64_t v_token_stride, void* query_out, void* key_out,
                        void* paged_kv_cache, int64_t page_stride, int64_t num_pages,
                        void* stream) {
  if (!plan) return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_run: null plan");
  const int64_t q_row = plan->num_heads * plan->head_dim;
  const int64_t k_row = plan->num_kv_heads * plan->head_dim;
  if (plan->slots) {
    if (page_stride < 2 * plan->page_size * k_row)
      return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_run: page_stride %lld < 2*page_size*H*D",
                  (long long)page_stride);
    const int E = plan->dtype == KVC_DTYPE_F32 ? 4 : 2;
    char* vc = paged_kv_cache ? (char*)paged_kv_cache + plan->page_size * k_row * E : nullptr;
    return kvc_rotary_pos_emb_and_cache(
        query, key, value, plan->positions, 4, plan->cos_sin_cache, plan->max_position, plan->nnz,
        plan->num_heads, plan->num_kv_heads, plan->head_dim, plan->rotary_dim, q_token_stride,
        k_token_stride, v_token_stride, query_out, key_out, q_row, k_row, paged_kv_cache, vc,
        plan->slots, 8, plan->page_size, page_stride, k_row, num_pages, plan->dtype, stream);
  }
  return kvc_rotary_pos_emb_and_append_paged(
      query, key, value, plan->batch_indices, plan->positions, plan->cos_sin_cache,
      plan->max_position, plan->nnz, plan->num_heads, plan->num_kv_heads, plan->head_dim,
      plan->rotary_dim, q_token_stride, k_token_stride, v_token_stride, query_out, key_out, q_row,
      k_row, paged_kv_cache, plan->kv_indices, plan->kv_indptr, plan->batch_size,
      plan->num_kv_indices, plan->page_size, page_stride, num_pages, plan->dtype, stream);
}

int kvc_rotary_plan_run_layers(const kvc_rotary_plan* plan, int64_t num_layers, const kvc_rotary_layer* layers,
                               int64_t q_token_stride, int64_t k_token_stride, int64_t v_token_stride,
                               int64_t page_stride, int64_t num_pages, int* one_launch, void* stream) {
  constexpr const char* fn = "kvc_rotary_plan_run_layers";
  if (one_launch) *one_launch = 0;
  if (!plan) return fail(KVC_ERR_INVALID_ARG, "%s: null plan", fn);
  if (num_layers < 0 || num_layers > 0xffff || (num_layers > 0 && !layers))
    return fail(KVC_ERR_INVALID_ARG, "%s: %lld layers", fn, (long long)num_layers);
  if (num_pages < 0 || page_stride < 0 || q_token_stride < 0 || k_token_stride < 0 || v_token_stride < 0)
    return fail(KVC_ERR_INVALID_ARG, "%s: negative size", fn);
  const int64_t q_row = plan->num_heads * plan->head_dim, k_row = plan->num_kv_heads * plan->head_dim;
  const int64_t E = plan->dtype == KVC_DTYPE_F32 ? 4 : 2, nnz = plan->nnz;
  const int64_t plane = plan->page_size * k_row;
  bool whole = plan->slots && num_layers > 1 && nnz > 0 && num_pages > 0 && page_stride >= 2 * plane;
  RopeLayer* const p = whole ? new (std::nothrow) RopeLayer[num_layers] : nullptr;
  whole = p != nullptr;
  for (int64_t l = 0; l < num_layers && whole; ++l) {
    const kvc_rotary_layer& y = layers[l];
    whole = y.query && y.key && y.value && y.query_out && y.paged_kv_cache;
    p[l] = RopeLayer{(const char*)y.query, (const char*)y.key, (const char*)y.value, (char*)y.query_out, (char*)y.key_out,
                     (char*)y.paged_kv_cache, (char*)y.paged_kv_cache + plane * E};
  }
  int rc = kLayerByLayer;
  if (whole && !layers_depend(p, num_layers,
                              {((nnz - 1) * q_token_stride + q_row) * E, ((nnz - 1) * k_token_stride + k_row) * E,
                               ((nnz - 1) * v_token_stride + k_row) * E, nnz * q_row * E, nnz * k_row * E,
                               ((num_pages - 1) * page_stride + 2 * plane) * E})) {
    const RopeGeom g{nnz, plan->num_heads, plan->num_kv_heads, plan->head_dim, plan->rotary_dim, plan->max_position,
                     q_token_stride, k_token_stride, v_token_stride, q_row, k_row, plan->dtype};
    const CacheGeom c{p->key_cache, p->value_cache, plan->slots, 8, nullptr, nullptr, nullptr, 0, 0,
                      plan->page_size, page_stride, k_row, num_pages};
    rc = run_rope(fn, p->query, p->key, p->value, p->query_out, p->key_out, plan->positions, 4,
                  plan->cos_sin_cache, g, &c, stream, p, num_layers);
  }
  delete[] p;
  if (rc != kLayerByLayer) {
    if (rc == KVC_OK && one_launch) *one_launch = 1;
    return rc;
  }
  for (int64_t l = 0; l < num_layers; ++l) {
    const kvc_rotary_layer& y = layers[l];
    rc = kvc_rotary_plan_run(plan, y.query, y.key, y.value, q_token_stride, k_token_stride, v_token_stride, y.query_out,
                             y.key_out, y.paged_kv_cache, page_stride, num_pages, stream);
    if (rc != KVC_OK) return rc;
  }
  return KVC_OK;
}

int kvc_rotary_plan_resolve_slots(kvc_rotary_plan* plan, int64_t* slots, void* stream) {
  if (!plan) return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_resolve_slots: null plan");
  const int rc = kvc::launch_resolve_slots("kvc_rotary_plan_resolve_slots", plan->batch_indices,
                                           plan->positions, plan->kv_indices, plan->kv_indptr,
                                           plan->batch_size, plan->num_kv_indices, plan->page_size,
                                           plan->nnz, slots, (hipStream_t)stream);
  if (rc == KVC_OK && plan->nnz > 0) plan->slots = slots;
  return rc;
}

int kvc_rotary_plan_set_slots(kvc_rotary_plan* plan, const int64_t* slots) {
  if (!plan) return fail(KVC_ERR_INVALID_ARG, "kvc_rotary_plan_set_slots: null plan");
  plan->slots = slots;
  return KVC_OK;
}

int kvc_rotary_plan_destroy(kvc_rotary_plan* plan) {
  delete plan;
  return KVC_OK;
}

}  // extern "C"
