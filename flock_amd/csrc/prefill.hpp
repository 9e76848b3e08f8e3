// Prefill kernel pieces: arguments, the schedule of key tiles over workgroups,
// the three-part bf16 split and the layout of split K/V tiles in LDS.
#pragma once

#include "common.hpp"

namespace flk {

constexpr int kRows = 128;      // query-head rows per q tile (4 blocks of 32)
constexpr int kBK = 64;         // keys per tile (2 halves of 32)
constexpr int kPThreads = 512;  // 8 waves: 4 row blocks x 2 key halves
constexpr uint32_t kMaxWG = 256;      // one workgroup per CU

// Where workgroup w of a kv head starts: key tile kt of the seq-th q tile (in
// the order of prefill_seq_qt). Workgroup w runs from start[w] up to start[w + 1].
struct PrefillStart {
  uint32_t seq, kt;
};

struct PrefillArgs {
  const float* q;
  const float* kcache;
  const float* vcache;
  float* o;
  float2* part_ml;   // [slot][kRows], slot = (2 w + last piece?) * n_kv_heads + kv head
  float* part_acc;   // [slot][kRows][D]
  uint32_t n_heads, n_kv_heads, group;
  uint32_t n_queries, pos0;
  uint32_t q_per_tile, n_qtiles;
  uint32_t wg_per_kvh;
  float scale_log2e;  // fr(1/sqrt(d) * log2(e)): scores in base-2 units
};

struct PrefillTable {
  PrefillStart start[kMaxWG + 1];
};

__host__ __device__ __forceinline__ uint32_t qtile_kt(uint32_t qt, uint32_t q_per_tile,
                                                      uint32_t n_queries, uint32_t pos0) {
  const uint32_t q_end = (qt + 1) * q_per_tile < n_queries ? (qt + 1) * q_per_tile : n_queries;
  return (uint32_t)(((uint64_t)pos0 + q_end + kBK - 1) / kBK);
}

// The q tiles in the order the workgroups take them: the heaviest, the
// lightest, the next heaviest, ... so that any stretch of a prompt's causal
// work cut out of the order holds about as many q tiles as any other.
__host__ __device__ __forceinline__ uint32_t prefill_seq_qt(uint32_t seq, uint32_t n_qtiles) {
  return seq & 1 ? seq >> 1 : n_qtiles - 1 - (seq >> 1);
}

// gfx9 buffer-descriptor word 3 for untyped 32-bit-element loads.
constexpr int kBufferWord3 = 0x00020000;

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t uint32x2 __attribute__((ext_vector_type(2)));

// ---- f32 as three bf16 -------------------------------------------------------
// x = s[0] + s[1] + s[2] exactly (each part takes the next 8 of the 24
// significand bits, rounded to nearest; both differences are exact). Parts of
// two values packed as the matrix operands want them.
__device__ __forceinline__ uint32_t bf16_pack(float a, float b) {
  const floatx2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&s)[3]) {
  s[0] = bf16_pack(a, b);
  a -= __builtin_bit_cast(float, s[0] << 16);
  b -= __builtin_bit_cast(float, s[0] & 0xffff0000u);
  s[1] = bf16_pack(a, b);
  a -= __builtin_bit_cast(float, s[1] << 16);
  b -= __builtin_bit_cast(float, s[1] & 0xffff0000u);
  s[2] = bf16_pack(a, b);
}

// acc += sum over k of a[k] b[k] with both operands in three parts: the six
// largest products, smallest first. A second part is at most
// 2^-8 of the value and a third 2^-17, so the three products left out are at most
// 2^-24 of |a| |b| together.
__device__ __forceinline__ void mfma_split(floatx16& acc, const uint32x4 (&a)[3],
                                           const uint32x4 (&b)[3]) {
  auto mul = [&](int i, int j) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[i]),
                                                  __builtin_bit_cast(bf16x8, b[j]), acc, 0, 0, 0);
  };
  mul(2, 0);
  mul(0, 2);
  mul(1, 1);
  mul(1, 0);
  mul(0, 1);
  mul(0, 0);
}

// ---- split tiles in LDS --------------------------------------------------------
// A tile is three planes (one per part) of 16-byte slots, each slot 8 bf16: one
// lane's share of a 16-deep matrix operand.
//   K: [64 keys][D / 8 slots]; slot c of a key holds dims 4c .. 4c + 3 and D/2 +
//      4c .. D/2 + 4c + 3 (so that the lanes that load a key's row read it as
//      contiguous float4s; q is permuted alike, and a dot product has no order).
//   V: [D channels][8 slots]; slot 2s + g of a channel holds keys 16s + 4g + {0
//      .. 3} and 16s + 8 + 4g + {0 .. 3}: the order in which lane half g holds
//      its scores of 16-key step s after S^T = K Q^T.
// The slot number is xored with bits of the row, so that any 8 (and 16, and 32)
// neighbouring lanes that read one slot of consecutive rows, or write a row, or
// write one slot of every other row, hit distinct banks.
template <int NS>
__device__ __forceinline__ int slot_swizzle(int row) {
  if constexpr (NS == 16) return (row & 15) ^ ((row >> 4) & 1);
  return (row & 7) ^ ((row >> 3) & 1) ^ (((row >> 4) & 1) << 1);
}

template <int D>
struct SplitTile {
  static constexpr int KS = D / 8;              // slots of a key
  static constexpr int kPlane = kBK * KS;       // slots of a plane (K and V alike)
  static constexpr int kSlots = 3 * kPlane;
  static constexpr int KP = kPlane / kPThreads;  // K slots (and V slots) a thread stages
};

}  // namespace flk
