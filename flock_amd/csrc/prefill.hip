// Causal GQA prefill attention as tiled flash attention on the bf16 matrix
// cores, in f32 precision (calls of little work: prefill_f32.hip).
//
// The reference (attention_prefill.wgsl:75-175) runs one workgroup per
// (query, head), streams every key of that query through scalar FMAs and two
// barrier-heavy tree reductions per 64-key tile. Here a work item is a "q
// tile" of up to 128 query-head rows that share one kv head ((128 / G) queries
// x the G heads of the group) and a range of its 64-key tiles.
//
// Arithmetic. f32 MFMAs run at 1/16 of the bf16 rate, so every operand is
// split into three bf16 parts that add up to it exactly, and a product takes
// six v_mfma_f32_32x32x16_bf16 (products of parts are exact in f32, sums are
// f32): 2.67 times the f32 rate. What is left out is at most 2^-24 of a
// product, half an ulp of it in f32 (of most significands below 2^-26); and an
// accumulator is rounded 6 times per 16 products instead of 16.
//
// Per 64-key tile, each of 8 waves owns 32 rows and one half (32 keys) of the
// tile; the two halves of a row keep separate online-softmax states and are
// combined through LDS when the item is done:
//   S^T = K Q^T     A = K [32 keys x 16 dims] from LDS, B = Q^T from registers
//                   (split once per item); out lane l, reg i holds
//                   S^T[key 8(i/4) + 4(l/32) + i%4][row l%32].
//   softmax         a query-head row lives in lanes l and l ^ 32: in-lane
//                   max/sum over 16 values. Running (m, l) per lane, no LDS.
//   O^T += V^T P^T  B = P^T split from the S^T registers (the key order inside
//                   a step is permuted alike on both operands); A = V^T from
//                   LDS. Lane l, reg i of channel block c holds channel 32c +
//                   8(i/4) + 4(l/32) + i%4 of row l%32.
// 32-row blocks: each 3 KB of K or V parts read from LDS serve 6 MFMAs, i.e.
// half of the LDS read rate; 16-row blocks would need all of it.
//
// What bounds it: the matrix cores and the power they draw. Over a 2048-token
// and an 8192-token prompt (16 / 8 heads of 128) MFMAs are busy 0.70 of the
// cycles, at 1.78 GHz of 2.4 (the f32 kernel: 0.75 of the cycles). Calls with
// their prologue, us, all of prefill on the f32 kernel -> here: 8192 tokens 2100 ->
// 1311, 2048 tokens 153.5 -> 120.8, 64 tokens at 32768 146 -> 114, 777 at 1000
// (32 / 8 heads of 64) 108 -> 72. Error against 64 bits: 5.2e-7 -> 4.5e-7, 3.9e-7 ->
// 3.2e-7, 7.3e-7 -> 5.7e-7, 5.7e-7 -> 4.0e-7.
//
// Staging. K and V tiles come through registers (requested a whole tile
// ahead), are split there, and go to a ring of three LDS tiles in the order
// K0 V0 K1 V1 ...: while tile u is used, u + 1 is split and stored, spread
// over the first half of u's matrix products; one barrier in the middle of
// each tile's use orders the ring. Between two barriers lie the second half
// of S, the softmax and the first half of PV, so the two waves of a SIMD drift
// apart and one's softmax runs under the other's matrix products. Rows past
// the last key are past the end of the loads' buffer descriptor and arrive as
// 0. Causal bound: query at absolute position p sees keys 0..p
// (attention_prefill.wgsl:90), applied per element.
//
// Scheduling: one workgroup per CU (workgroup id = kv head + n_kv_heads * w, so
// with 8 kv heads the workgroups of one kv head share an XCD and its L2). A kv
// head's key tiles, q tile after q tile in the order heaviest, lightest, next
// heaviest ..., are cut into equal runs, one per workgroup (the host's table
// `start`), whatever the shape: a prompt's causal triangle, a chunk onto a long
// cache. Pieces of q tiles that were cut go through partials, which
// prefill_merge_kernel combines.
#include "prefill.hpp"

namespace flk {

// ---- inputs that three bf16 parts do not cover -----------------------------------
// A row of an item is formed again in plain f32 (row_f32) where the parts lose
// something; what decides is the row's own q and its own result:
// - an output that is no finite number: an infinity or NaN in q, K or V, or a
//   magnitude that bf16 rounds to infinity, splits into infinite - infinite. What
//   f32 arithmetic makes of such inputs (a -inf score weighs nothing, an infinite v
//   gives an infinite output) is formed here.
// - q with an element other than 0 below kTinyQ, or one of at least kLargeQ. Parts end
//   at 2^-133, bf16's smallest number (the matrix cores keep it), so a value of less
//   than 2^-110 loses up to 2^-134, which costs a score that times the other factor:
//   with no part of q lost, at most D 2^-134 kLargeQ = 2^-27.
// - a normalised output other than 0 below kTinyOutput: lost parts of v cost it up to
//   2^-134, i.e. up to 2^-26 of itself above that. (A v below 2^-134 counts as 0
//   where no output of the row shows it.)
// Weights lose as little: one below 2^-110 of the row's largest is off by up to 2^-134
// of that (and one below 2^-126 is 0, as in the f32 kernel).
// A v that is not finite past a row's last key reaches the row too (0 x infinite):
// its result is the one of its own keys, but its last bits may differ.
constexpr float kTinyOutput = 0x1p-108f, kTinyQ = 0x1p-110f, kLargeQ = 0x1p100f;

// What a workgroup's waves tell each other about such rows, in LDS.
struct Redo {
  uint32_t any;              // some row is to be formed again
  uint32_t bad[kRows / 32];  // which
  uint32_t no_nan_key;       // ~(the first key of the item with a NaN in K)
};

// One row's attention over keys key0 .. key1 - 1 in plain f32 by one wave: lane
// = key for the scores, lane = channels for the sums. Returns (m, l) and, in
// lane l, channels l, l + 64, ... of the unnormalised sum.
template <int D>
__device__ void row_f32(const PrefillArgs& a, uint32_t lane, const float* qrow, uint32_t kvh,
                        uint32_t key0, uint32_t key1, float& m, float& l,
                        float (&acc)[D / 64]) {
  const size_t stride = (size_t)a.n_kv_heads * D;
  const float* kb = a.kcache + (size_t)kvh * D;
  const float* vb = a.vcache + (size_t)kvh * D;
  m = -1e30f;
  l = 0.f;
#pragma unroll
  for (int c = 0; c < D / 64; c++) acc[c] = 0.f;
  for (uint32_t k0 = key0; k0 < key1; k0 += 64) {
    const uint32_t key = k0 + lane;
    float s = -INFINITY;
    if (key < key1) {
      const float4* kr = reinterpret_cast<const float4*>(kb + key * stride);
      const float4* qr = reinterpret_cast<const float4*>(qrow);
      s = 0.f;
#pragma unroll 4
      for (int c = 0; c < D / 4; c++) {
        const float4 k = kr[c], q = qr[c];
        s = fmaf(k.x, q.x * a.scale_log2e, s);
        s = fmaf(k.y, q.y * a.scale_log2e, s);
        s = fmaf(k.z, q.z * a.scale_log2e, s);
        s = fmaf(k.w, q.w * a.scale_log2e, s);
      }
    }
    float mx = s;
#pragma unroll
    for (int x = 32; x >= 1; x >>= 1) mx = fmaxf(mx, shfl_xor(mx, x));
    if (mx > m) {  // uniform
      const float corr = __builtin_amdgcn_exp2f(m - mx);
      l *= corr;
#pragma unroll
      for (int c = 0; c < D / 64; c++) acc[c] *= corr;
      m = mx;
    }
    const float p = __builtin_amdgcn_exp2f(s - m);
    float sum = p;
#pragma unroll
    for (int x = 32; x >= 1; x >>= 1) sum += shfl_xor(sum, x);
    l += sum;
    float blk[D / 64];  // of these keys: a long sum is rounded once per 64 keys
#pragma unroll
    for (int c = 0; c < D / 64; c++) blk[c] = 0.f;
    const uint32_t n = min(key1 - k0, 64u);
    for (uint32_t j0 = 0; j0 < n; j0 += 8) {
      float v[8][D / 64];
#pragma unroll
      for (int j = 0; j < 8; j++)
#pragma unroll
        for (int c = 0; c < D / 64; c++)
          v[j][c] = vb[min(k0 + j0 + j, key1 - 1) * stride + 64 * c + lane];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float pj = __builtin_bit_cast(
            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), j0 + j));
#pragma unroll
        for (int c = 0; c < D / 64; c++)
          blk[c] = j0 + j < n ? fmaf(pj, v[j][c], blk[c]) : blk[c];
      }
    }
#pragma unroll
    for (int c = 0; c < D / 64; c++) acc[c] += blk[c];
    if (l != l) return;  // NaN in every channel, whatever follows
  }
}

// Where redo_rows puts row r's channels and (m, l): in two tiles of the ring.
template <int D>
__device__ __forceinline__ float* row_lds(uint32x4* const (&buf)[2], uint32_t r) {
  return reinterpret_cast<float*>(buf[r / (kRows / 2)]) + r % (kRows / 2) * D;
}
template <int D>
__device__ __forceinline__ float2* ml_lds(uint32x4* const (&buf)[2]) {
  static_assert(kRows / 2 * D / 4 + kRows / 2 <= SplitTile<D>::kSlots, "rows and (m, l) fit");
  return reinterpret_cast<float2*>(buf[1] + kRows / 2 * D / 4);
}

// Forms the rows of `s` again, into LDS: channels (divided by l when `final`) and
// (m, l). Rows that see a NaN in K are NaN already and leave s, so that a NaN token
// costs little; other rows cost a wave the reads of all their keys. 16 / 8 heads of
// 128, us, 2048 and 8192 tokens: 117, 1270; a NaN token half way 130, 1470; an infinite
// v that every row sees 2940, 55000 (the f32 kernel, which that does not slow: 157,
// 2100).
template <int D>
__device__ void redo_rows(const PrefillArgs& a, Redo& s, uint32x4* const (&buf)[2], uint32_t kvh,
                          uint32_t qt, uint32_t kt0, uint32_t kt1, bool final) {
  uint32_t tid = threadIdx.x;  // opaque: nothing of this is formed for every item
  asm volatile("" : "+v"(tid));
  const uint32_t lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t key0 = kt0 * kBK, key1 = min(kt1 * kBK, a.pos0 + a.n_queries);
  constexpr int CH = D / 4;
  uint32_t nan_key = ~0u;
#pragma unroll 4
  for (uint32_t key = key0 + tid / CH; key < key1; key += kPThreads / CH) {
    const float4 k = *reinterpret_cast<const float4*>(
        a.kcache + ((size_t)key * a.n_kv_heads + kvh) * D + 4 * (tid % CH));
    if (k.x != k.x || k.y != k.y || k.z != k.z || k.w != k.w) nan_key = min(nan_key, key);
  }
  if (nan_key != ~0u) atomicMax(&s.no_nan_key, ~nan_key);
  __syncthreads();
  nan_key = ~s.no_nan_key;
  for (uint32_t r = wave; r < a.q_per_tile * a.group; r += kPThreads / 64) {
    const uint32_t bit = 1u << r % 32, pos = a.pos0 + qt * a.q_per_tile + r / a.group;
    if (!(s.bad[r / 32] & bit)) continue;
    if (pos >= nan_key) {
      if (lane == 0) atomicAnd(&s.bad[r / 32], ~bit);
      continue;
    }
    const float* q = a.q + ((size_t)(pos - a.pos0) * a.n_heads + kvh * a.group + r % a.group) * D;
    float m, l, acc[D / 64];
    row_f32<D>(a, lane, q, kvh, key0, min(key1, pos + 1), m, l, acc);
#pragma unroll
    for (int i = 0; i < D / 64; i++)
      row_lds<D>(buf, r)[64 * i + lane] = final ? acc[i] / l : acc[i];
    if (lane == 0) ml_lds<D>(buf)[r] = make_float2(m, l);
  }
  __syncthreads();
}

// Key tiles on their way to LDS: this thread's share of one K and one V tile.
template <int D>
struct Staged {
  using T = SplitTile<D>;
  uint32x4 k[T::KP][2];    // slot i: float4 c and D/8 + c of a key
  float v[T::KP][8];       // channel i of 8 keys
};

template <int D>
struct TileLoader {
  using T = SplitTile<D>;
  uint32_t koff, voff;  // this thread's first bytes within a tile
  int kdst, vdst;       // its first slots within a plane
  uint32_t row_bytes;

  __device__ __forceinline__ explicit TileLoader(uint32_t rb) : row_bytes(rb) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // K: slot c of key tid / KS (and of key 32 + that, which swizzles alike).
    const int c = tid % T::KS, key = tid / T::KS;
    koff = key * rb + 16 * c;
    kdst = key * T::KS + (c ^ slot_swizzle<T::KS>(key));
    // V: wave w has slot w of every channel; lane l channels KP l ...
    voff = (16 * (wave >> 1) + 4 * (wave & 1)) * rb + 4 * T::KP * lane;
    vdst = T::KP * lane * 8 + (wave ^ slot_swizzle<8>(T::KP * lane));
  }
  __device__ __forceinline__ int k_slot(int i) const { return kdst + 32 * T::KS * i; }
  // The odd neighbour of an even channel: the next row, the lowest slot bit
  // flipped.
  __device__ __forceinline__ int v_slot(int i) const { return i ? (vdst ^ 1) + 8 : vdst; }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const PrefillArgs& a, const float* cache,
                                                         uint32_t kvh, uint32_t kt) const {
    const uint32_t key0 = kt * kBK;
    const uint32_t rows = min(a.pos0 + a.n_queries - key0, (uint32_t)kBK);
    const size_t base = (size_t)key0 * row_bytes + (size_t)kvh * D * 4;
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(reinterpret_cast<const char*>(cache) + base), 0,
        (rows - 1) * row_bytes + D * 4, kBufferWord3);
  }
  // The offsets are made opaque so that their sums with the row steps are
  // formed at each use and not kept in registers.
  __device__ __forceinline__ void load_k(Staged<D>& s, const PrefillArgs& a, uint32_t kvh,
                                         uint32_t kt) const {
    const __amdgpu_buffer_rsrc_t r = rsrc(a, a.kcache, kvh, kt);
    uint32_t off = koff;
    asm volatile("" : "+v"(off));
#pragma unroll
    for (int i = 0; i < T::KP; i++) {
      s.k[i][0] = __builtin_amdgcn_raw_buffer_load_b128(r, off + 32 * i * row_bytes, 0, 0);
      s.k[i][1] = __builtin_amdgcn_raw_buffer_load_b128(r, off + 32 * i * row_bytes + 2 * D, 0, 0);
    }
  }
  __device__ __forceinline__ void load_v(Staged<D>& s, const PrefillArgs& a, uint32_t kvh,
                                         uint32_t kt) const {
    const __amdgpu_buffer_rsrc_t r = rsrc(a, a.vcache, kvh, kt);
    uint32_t off = voff;
    asm volatile("" : "+v"(off));
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint32_t o = off + ((j & 3) + 8 * (j >> 2)) * row_bytes;
      if constexpr (T::KP == 2) {
        const uint32x2 w = __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0);
        s.v[0][j] = __builtin_bit_cast(float, (uint32_t)w.x);
        s.v[1][j] = __builtin_bit_cast(float, (uint32_t)w.y);
      } else {
        s.v[0][j] = __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0));
      }
    }
  }
};

// Step n = 4i + e of staging a tile: splits values 2e, 2e + 1 of this thread's
// slot i; the slot's last step stores it.
template <int D, bool V>
__device__ __forceinline__ void stage_step(int n, const Staged<D>& s, const TileLoader<D>& ld,
                                           uint32x4* dst, uint32x4 (&w)[3]) {
  const int i = n / 4, e = n % 4;
  float x, y;
  if (V) {
    x = s.v[i][2 * e];
    y = s.v[i][2 * e + 1];
  } else {
    x = __builtin_bit_cast(float, (uint32_t)s.k[i][e / 2][2 * (e % 2)]);
    y = __builtin_bit_cast(float, (uint32_t)s.k[i][e / 2][2 * (e % 2) + 1]);
  }
  uint32_t p[3];
  split_pair(x, y, p);
#pragma unroll
  for (int k = 0; k < 3; k++) w[k][e] = p[k];
  if (e == 3) {
#pragma unroll
    for (int k = 0; k < 3; k++)
      dst[k * SplitTile<D>::kPlane + (V ? ld.v_slot(i) : ld.k_slot(i))] = w[k];
  }
}

#define FLK_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

// A lane's row of a q tile: r -> (query, head).
template <int D>
struct QRow {
  uint32_t qi, h;
  bool ok;

  __device__ __forceinline__ QRow(const PrefillArgs& a, uint32_t kvh, uint32_t qt) {
    const uint32_t r = ((threadIdx.x >> 6) & 3) * 32 + (threadIdx.x & 31);
    qi = qt * a.q_per_tile + r / a.group;
    h = kvh * a.group + r % a.group;
    ok = r < a.q_per_tile * a.group && qi < a.n_queries;
    if (!ok) {  // reads the tile's first row, writes nothing
      qi = qt * a.q_per_tile;
      h = kvh * a.group;
    }
  }
  __device__ __forceinline__ size_t offset(const PrefillArgs& a) const {
    return ((size_t)qi * a.n_heads + h) * D;
  }
  // Dims of slots 2j + lg.
  __device__ __forceinline__ void fetch(float4 (&q)[D / 8], const PrefillArgs& a) const {
    const int lg = (threadIdx.x >> 5) & 1;
    const float4* src = reinterpret_cast<const float4*>(a.q + offset(a));
#pragma unroll
    for (int j = 0; j < D / 16; j++) {
      q[2 * j] = src[2 * j + lg];
      q[2 * j + 1] = src[D / 8 + 2 * j + lg];
    }
  }
};

// What a workgroup carries from item to item: the ring (K of the current tile,
// its V, K of the next), and the loads in flight.
template <int D>
struct Pipe {
  uint32x4 *bk, *bv, *bn;
  Staged<D> st;
  float4 q[D / 8];
};

// Key tiles [kt0, kt1) of q tile qt of kv head kvh; writes o rows (normalised)
// when `final`, else the partial of `slot`. The caller has put tile kt0's K into
// p.bk (all but the barrier) and requested its V and the q rows. Under the last
// tile the next item's first key tile (nxt_kt) goes the same way, and q tile
// nxt_qt's rows are requested under the combine; without a next item the caller
// names a tile of this one.
template <int D>
__device__ __forceinline__ void run_item(const PrefillArgs& a, Pipe<D>& p, Redo* redo, uint32_t kvh,
                                         uint32_t qt, uint32_t kt0, uint32_t kt1, bool final,
                                         size_t slot, const TileLoader<D>& ld, uint32_t nxt_qt,
                                         uint32_t nxt_kt) {
  using T = SplitTile<D>;
  constexpr int NG = D / 16;  // groups of 6 products of S, and of PV
  constexpr int CB = D / 32;  // channel blocks of O^T
  constexpr int SG = NG / 4;  // groups under which a tile is split and stored
  constexpr int BG = SG;      // group after which the barrier comes
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = wave >> 2;  // which 32 keys of every tile this wave takes
  const int lc = lane & 31, lg = lane >> 5;
  const uint32_t q0 = qt * a.q_per_tile;
  const uint32_t r = (wave & 3) * 32 + lc;
  const QRow<D> row(a, kvh, qt);
  const uint32_t qpos = a.pos0 + row.qi;
  const bool row_ok = row.ok;
  uint32x4 *bk = p.bk, *bv = p.bv, *bn = p.bn;
  Staged<D>& st = p.st;
  uint32x4 w[3];
  // The row's q, pre-multiplied by scale * log2(e) so that S^T comes out in
  // base-2 units, split.
  uint32x4 qf[NG][3];
#pragma unroll
  for (int j = 0; j < NG; j++) {
    const float4 x = p.q[2 * j], y = p.q[2 * j + 1];
    const float e[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint32_t u[3];
      split_pair(e[2 * i] * a.scale_log2e, e[2 * i + 1] * a.scale_log2e, u);
#pragma unroll
      for (int k = 0; k < 3; k++) qf[j][k][i] = u[k];
    }
  }
  lds_barrier();  // before the branch below, or every wave waits for the slowest q
  // 2^-63 <= |q| < 2^65 has top exponent bits 01 or 10; a row with others (or
  // zeros) is read again and looked at. Each of the row's two waves takes half of q.
  uint32_t q_mid = ~0u;  // bits 14 and 30: the top two exponent bits differ everywhere
#pragma unroll
  for (int h = 0; h < 2; h++)
    if (h == half) {  // uniform
#pragma unroll
      for (int j = 0; j < NG / 2; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const uint32_t u = qf[h * NG / 2 + j][0][i];
          q_mid &= u ^ (u << 1);
        }
    }
  bool q_out = false;
  if (__builtin_amdgcn_ballot_w64((q_mid & 0x40004000u) != 0x40004000u) != 0) {  // uniform
    float4 q[D / 8];
    row.fetch(q, a);
    float least = 1.f, most = 0.f;  // magnitudes other than 0; a NaN stays in `most`
#pragma unroll
    for (int j = 0; j < D / 8; j++) {
      const float e[4] = {q[j].x, q[j].y, q[j].z, q[j].w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float x = fabsf(e[i] * a.scale_log2e);
        least = fminf(least, x != 0.f ? x : 1.f);
        most = __builtin_elementwise_maximum(most, x);
      }
    }
    q_out = least < kTinyQ || !(most < kLargeQ);
  }

  floatx16 oacc[CB];
#pragma unroll
  for (int c = 0; c < CB; c++)
#pragma unroll
    for (int i = 0; i < 16; i++) oacc[c][i] = 0.f;
  // Running reference m_run (log2 units; finite, so that a masked key's
  // weight exp2(-inf - m_run) is exactly 0) and this lane's share of the
  // denominator (its keys only).
  float m_run = -1e30f, l_run = 0.f;

  // A tile needs no causal mask when its last key is at or before the q
  // tile's first query position and every row of the q tile is live.
  const bool all_rows = a.q_per_tile * a.group == kRows && q0 + a.q_per_tile <= a.n_queries;
  // Byte offsets of this lane's slot 0 + lg of its K row, V row within a plane;
  // slot 2x + lg is that offset ^ 32x (the rows are aligned to their length).
  const uint32_t kaddr = 16 * ((half * 32 + lc) * T::KS + (lg ^ slot_swizzle<T::KS>(lc)));
  const uint32_t vaddr = 16 * (lc * 8 + (lg ^ slot_swizzle<8>(lc))) ^ (64 * half);
  uint32_t kaddr_o = kaddr;
  auto read_k = [&](uint32x4 (&f)[3], int j) {
    const uint32x4* p = reinterpret_cast<const uint32x4*>(
        reinterpret_cast<const char*>(bk) + (kaddr_o ^ (32 * j)));
#pragma unroll
    for (int k = 0; k < 3; k++) f[k] = p[k * T::kPlane];
  };
  // PV group n: channel block n % CB, 16-key step n / CB.
  auto read_v = [&](uint32x4 (&f)[3], int n) {
    const uint32x4* p = reinterpret_cast<const uint32x4*>(
        reinterpret_cast<const char*>(bv) + (vaddr ^ (32 * (n / CB)))) + (n % CB) * 256;
#pragma unroll
    for (int k = 0; k < 3; k++) f[k] = p[k * T::kPlane];
  };

#pragma unroll 1
  for (uint32_t kt = kt0; kt < kt1; kt++) {
    const uint32_t key0 = kt * kBK;
    const uint32_t kt_1 = kt + 1 < kt1 ? kt + 1 : nxt_kt;
    kaddr_o = kaddr;  // opaque: its xors are formed at each use
    asm volatile("" : "+v"(kaddr_o));
    // ---- S^T = K Q^T, V split and stored under its first half ----------------------
    floatx16 s;
#pragma unroll
    for (int i = 0; i < 16; i++) s[i] = 0.f;
    uint32x4 f[2][3];
    read_k(f[0], 0);
    FLK_SCHED_FENCE();
#pragma unroll
    for (int j = 0; j < NG; j++) {
      if (j + 1 < NG) read_k(f[(j + 1) & 1], j + 1);
      mfma_split(s, f[j & 1], qf[j]);
      if (j < SG) {
#pragma unroll
        for (int e = 0; e < 4; e++) stage_step<D, true>(4 * j + e, st, ld, bv, w);
      }
      if (j == BG) {
        ld.load_k(st, a, kvh, kt_1);
        lds_barrier();
      }
      FLK_SCHED_FENCE();
    }

    // ---- online softmax of this lane's row (base 2) ----------------------------
    // Scores are base-2 already (q carries scale * log2(e)), so every weight is
    // one v_exp_f32 against the reference m_run. The reference moves only when
    // some score of the wave exceeds it by more than 8 (a factor 256): the
    // check needs only each lane's own 16 scores, and the row's maximum across
    // its two lanes is formed only then (rarely after the first tile).
    // Otherwise the weights are taken against the old reference -- each at
    // most 256 -- and nothing is rescaled. Tiles wholly below the causal
    // diagonal with every row live skip the mask.
    if (!(all_rows && key0 + kBK - 1 <= a.pos0 + q0)) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const uint32_t key = key0 + half * 32 + 8 * (i / 4) + 4 * lg + i % 4;
        s[i] = row_ok && key <= qpos ? s[i] : -INFINITY;
      }
    }
    float lmx = s[0];
#pragma unroll
    for (int i = 1; i < 16; i++) lmx = fmaxf(lmx, s[i]);
    if (__builtin_amdgcn_ballot_w64(lmx > m_run + 8.f) != 0) {  // uniform branch
      // Only rows whose own maximum passed the threshold move their reference;
      // the others keep it and are multiplied by exactly 1, so a row's result
      // depends on its own keys only (causality holds bit for bit, but for a v
      // that is not finite past the row's last key: row_f32).
      const float mx = max_xor<32>(lmx);
      const bool up = mx > m_run + 8.f;
      const float corr = up ? __builtin_amdgcn_exp2f(m_run - mx) : 1.f;
      l_run *= corr;
#pragma unroll
      for (int c = 0; c < CB; c++) oacc[c] *= corr;
      m_run = up ? mx : m_run;
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
      s[i] = __builtin_amdgcn_exp2f(s[i] - m_run);
      l_run += s[i];
    }
    uint32x4 pf[2][3];
    auto split_p = [&](int e) {  // weights 2e, 2e + 1
      uint32_t p[3];
      split_pair(s[2 * e], s[2 * e + 1], p);
#pragma unroll
      for (int k = 0; k < 3; k++) pf[e / 4][k][e % 4] = p[k];
    };
    uint32x4 g[2][3];
    read_v(g[0], 0);
#pragma unroll
    for (int e = 0; e < 4; e++) split_p(e);

    // ---- O^T += V^T P^T; under its first half (step 0) the weights of step 1 are
    // split, and the next K is split and stored --------------------------------------
#pragma unroll
    for (int n = 0; n < NG; n++) {
      if (n + 1 < NG) read_v(g[(n + 1) & 1], n + 1);
      mfma_split(oacc[n % CB], g[n & 1], pf[n / CB]);
      if (n < CB) {
#pragma unroll
        for (int e = 0; e < 4 / CB; e++) split_p(4 + n * (4 / CB) + e);
      }
      if (n < SG) {
#pragma unroll
        for (int e = 0; e < 4; e++) stage_step<D, false>(4 * n + e, st, ld, bn, w);
      }
      if (n == BG) {
        ld.load_v(st, a, kvh, kt_1);
        lds_barrier();
      }
      FLK_SCHED_FENCE();
    }
    uint32x4* t = bk;
    bk = bn;
    bn = bv;
    bv = t;
  }

  p.bk = bk;
  p.bv = bv;
  p.bn = bn;
  QRow<D>(a, kvh, nxt_qt).fetch(p.q, a);
  l_run = sum_xor<32>(l_run);  // the row's two lanes
  // ---- combine the two key halves of each row through LDS --------------------
  // Each half hands the other its channel blocks of the other's share (half 0
  // finishes blocks 0 .. CB/2 - 1, half 1 the rest) and its (m, l), through the
  // two tiles of the ring that do not hold the next item's K.
  constexpr int HB = CB / 2;
  static_assert(HB * 1024 + 128 <= T::kSlots, "half the exchange and (m, l) fit a tile");
  lds_barrier();  // every wave is done with the ring
  float2* ml_x = reinterpret_cast<float2*>(bn + HB * 1024);  // [half][kRows]
  floatx16 mine[HB];
#pragma unroll
  for (int c = 0; c < HB; c++) {
    const floatx16 give = half ? oacc[c] : oacc[HB + c];
    mine[c] = half ? oacc[HB + c] : oacc[c];
#pragma unroll
    for (int j = 0; j < 4; j++)
      (half ? bn : bv)[(((wave & 3) * HB + c) * 4 + j) * 64 + lane] = __builtin_bit_cast(
          uint32x4, make_float4(give[4 * j], give[4 * j + 1], give[4 * j + 2], give[4 * j + 3]));
  }
  if (lg == 0) ml_x[half * kRows + r] = make_float2(m_run, l_run);
  if (threadIdx.x < sizeof(Redo) / 4)
    reinterpret_cast<uint32_t*>(redo)[threadIdx.x] = 0;
  lds_barrier();
  const float2 ml2 = ml_x[(1 - half) * kRows + r];
  const float M = fmaxf(m_run, ml2.x);
  // A half that saw no key of this row still holds the initial reference
  // (-1e30, l = 0): its weight exp2(-1e30 - M) is 0. A row with no key in the
  // item at all has both at the initial reference and sums of 0.
  const float w1 = __builtin_amdgcn_exp2f(m_run - M);
  const float w2 = __builtin_amdgcn_exp2f(ml2.x - M);
  const float L = l_run * w1 + ml2.y * w2;
  // Stored as they come, and looked at meanwhile: stores held back until all were
  // looked at cost 0.5 us per item.
  float* dst;
  if (final) {
    dst = a.o + row.offset(a);
  } else {
    dst = a.part_acc + (slot * kRows + r) * D;
    if (lg == 0 && half == 0) a.part_ml[slot * kRows + r] = make_float2(M, L);
  }
  dst += 32 * HB * half + 4 * lg;  // channel 32c + 8j of this lane at 32c + 8j
  float least = INFINITY, most = 0.f;  // magnitudes; a NaN stays in `most`
#pragma unroll
  for (int c = 0; c < HB; c++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float4 x = __builtin_bit_cast(
          float4, (half ? bv : bn)[(((wave & 3) * HB + c) * 4 + j) * 64 + lane]);
      float4 v = make_float4(mine[c][4 * j] * w1 + x.x * w2, mine[c][4 * j + 1] * w1 + x.y * w2,
                             mine[c][4 * j + 2] * w1 + x.z * w2,
                             mine[c][4 * j + 3] * w1 + x.w * w2);
      if (final) v = make_float4(v.x / L, v.y / L, v.z / L, v.w / L);
      const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        least = fminf(least, fabsf(e[i]));
        most = __builtin_elementwise_maximum(most, fabsf(e[i]));
      }
      if (row_ok || !final) *reinterpret_cast<float4*>(dst + 32 * c + 8 * j) = v;
    }
  const float tiny = final ? kTinyOutput : kTinyOutput * L;
  const bool look = row_ok && (q_out || !(most < INFINITY) || !(least >= tiny));
  if (__builtin_amdgcn_ballot_w64(look) != 0) {  // uniform
    least = INFINITY;  // of the others than 0
#pragma unroll
    for (int c = 0; c < HB; c++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float4 v = *reinterpret_cast<const float4*>(dst + 32 * c + 8 * j);
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) least = fminf(least, e[i] != 0.f ? fabsf(e[i]) : INFINITY);
      }
    if (row_ok && (q_out || !(most < INFINITY) || least < tiny)) {
      atomicOr(&redo->bad[wave & 3], 1u << lc);
      redo->any = 1;
    }
  }
  __syncthreads();  // every wave is done with the exchange (the next item's V goes there)
  if (redo->any) {  // uniform
    uint32x4* const buf[2] = {bv, bn};
    redo_rows<D>(a, *redo, buf, kvh, qt, kt0, kt1, final);
    if (redo->bad[wave & 3] >> lc & 1) {
      const float* x = row_lds<D>(buf, r) + 32 * HB * half + 4 * lg;
#pragma unroll
      for (int c = 0; c < HB; c++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          *reinterpret_cast<float4*>(dst + 32 * c + 8 * j) =
              *reinterpret_cast<const float4*>(x + 32 * c + 8 * j);
      if (!final && lg == 0 && half == 0) a.part_ml[slot * kRows + r] = ml_lds<D>(buf)[r];
    }
    // Requested again, so that nothing else is held over redo_rows.
    QRow<D>(a, kvh, nxt_qt).fetch(p.q, a);
    ld.load_v(st, a, kvh, nxt_kt);
  }
}

template <int D>
__global__ __launch_bounds__(kPThreads, 2) void prefill_kernel(PrefillArgs a, PrefillTable tab) {
  __shared__ uint32x4 lds[3 * SplitTile<D>::kSlots];
  __shared__ Redo redo;
  const uint32_t kvh = blockIdx.x % a.n_kv_heads;
  const uint32_t w = blockIdx.x / a.n_kv_heads;
  const TileLoader<D> ld(a.n_kv_heads * D * 4);
  const PrefillStart s0 = tab.start[w], s1 = tab.start[w + 1];
  uint32_t seq = s0.seq, kt0 = s0.kt;
  auto live = [&](uint32_t x, uint32_t kt) { return x < s1.seq || (x == s1.seq && kt < s1.kt); };
  if (!live(seq, kt0)) return;  // uniform
  Pipe<D> p;
  p.bk = lds;
  p.bv = lds + SplitTile<D>::kSlots;
  p.bn = lds + 2 * SplitTile<D>::kSlots;
  ld.load_k(p.st, a, kvh, kt0);
  QRow<D>(a, kvh, prefill_seq_qt(seq, a.n_qtiles)).fetch(p.q, a);
  ld.load_v(p.st, a, kvh, kt0);
  uint32x4 t[3];
#pragma unroll
  for (int n = 0; n < 4 * SplitTile<D>::KP; n++) stage_step<D, false>(n, p.st, ld, p.bk, t);
  while (live(seq, kt0)) {
    const uint32_t qt = prefill_seq_qt(seq, a.n_qtiles);
    const uint32_t n_kt = qtile_kt(qt, a.q_per_tile, a.n_queries, a.pos0);
    const uint32_t kt1 = seq == s1.seq ? s1.kt : n_kt;
    // A workgroup's first piece of a cut q tile has slot 2w, its last 2w + 1.
    const size_t slot = (size_t)(2 * w + (seq != s0.seq ? 1 : 0)) * a.n_kv_heads + kvh;
    const bool more = live(seq + 1, 0);
    run_item<D>(a, p, &redo, kvh, qt, kt0, kt1, kt0 == 0 && kt1 == n_kt, slot, ld,
                more ? prefill_seq_qt(seq + 1, a.n_qtiles) : qt, more ? 0 : kt0);
    seq++;
    kt0 = 0;
  }
}

// One workgroup per (kv head, workgroup w of prefill_kernel, 256 / (D/4)
// rows); D/4 lanes per row, each owning a float4 of channels. If a cut q tile
// starts in w, combines its pieces (w's last or only one, then the first of w +
// 1, w + 2, ... until the tile ends) with log-sum-exp weights in one pass: the
// pieces go in rounds of kPMergeBatch whose loads are all issued first (indices
// past the last piece reload it and get weight 0, so every load is
// unconditional), then folded against a running maximum.
constexpr int kPMergeBatch = 8;
template <int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a, PrefillTable tab) {
  constexpr int LPR = D / 4;
  constexpr int RPB = 256 / LPR;   // rows per block
  const uint32_t kvh = blockIdx.x;
  const uint32_t w = blockIdx.y;
  const uint32_t seq = tab.start[w + 1].seq;
  const PrefillStart s0 = tab.start[w];
  // Cut at the end of w, and started in w.
  if (tab.start[w + 1].kt == 0 || (s0.seq == seq && s0.kt != 0)) return;
  const uint32_t first = 2 * w + (s0.seq != seq ? 1 : 0);
  uint32_t ns = 2;
  while (tab.start[w + ns].seq == seq && tab.start[w + ns].kt != 0) ns++;
  const uint32_t qt = prefill_seq_qt(seq, a.n_qtiles);
  const uint32_t r = blockIdx.z * RPB + threadIdx.x / LPR;
  const int c = threadIdx.x % LPR;
  const uint32_t qi = qt * a.q_per_tile + r / a.group;
  if (r >= a.q_per_tile * a.group || qi >= a.n_queries) return;
  const uint32_t h = kvh * a.group + r % a.group;
  float M = -INFINITY, L = 0.f;
  float4 A = make_float4(0.f, 0.f, 0.f, 0.f);
  for (uint32_t p0 = 0; p0 < ns; p0 += kPMergeBatch) {
    float2 ml[kPMergeBatch];
    float4 pa[kPMergeBatch];
#pragma unroll
    for (int i = 0; i < kPMergeBatch; i++) {
      const uint32_t sp = min(p0 + i, ns - 1);
      const size_t slot = (size_t)(sp == 0 ? first : 2 * (w + sp)) * a.n_kv_heads + kvh;
      ml[i] = a.part_ml[slot * kRows + r];
      pa[i] = reinterpret_cast<const float4*>(a.part_acc + (slot * kRows + r) * D)[c];
    }
#pragma unroll
    for (int i = 0; i < kPMergeBatch; i++)
      if (p0 + i >= ns) {  // a reloaded piece: weight 0
        ml[i].x = -INFINITY;
        pa[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    float mx = M;
#pragma unroll
    for (int i = 0; i < kPMergeBatch; i++) mx = fmaxf(mx, ml[i].x);  // piece p0's is no -inf
    const float wo = __builtin_amdgcn_exp2f(M - mx);  // m is in log2 units; exp2(-inf) = 0
    L *= wo;
    A.x *= wo;
    A.y *= wo;
    A.z *= wo;
    A.w *= wo;
#pragma unroll
    for (int i = 0; i < kPMergeBatch; i++) {
      const float wt = __builtin_amdgcn_exp2f(ml[i].x - mx);
      L = fmaf(ml[i].y, wt, L);
      A.x = fmaf(pa[i].x, wt, A.x);
      A.y = fmaf(pa[i].y, wt, A.y);
      A.z = fmaf(pa[i].z, wt, A.z);
      A.w = fmaf(pa[i].w, wt, A.w);
    }
    M = mx;
  }
  float4* dst = reinterpret_cast<float4*>(a.o + ((size_t)qi * a.n_heads + h) * D);
  dst[c] = make_float4(A.x / L, A.y / L, A.z / L, A.w / L);
}

// ------------------------------------------------------------------ plan ----
static uint64_t prefill_max_wg(uint32_t n_kv_heads) {
  return n_kv_heads < kMaxWG ? kMaxWG / n_kv_heads : 1;
}

// Estimated time (us) of the f32 kernel under its plan: 1-tile items cost 5 +
// 4.4 (head_dim 64: 3.5 + 2.5), a merge 5; more workgroups than CUs run in rounds.
// Closer where that is known to mislead, at head_dim 128 (one workgroup per CU) and
// with more kv heads than half the CUs: pairs of q tiles count by their halves (the
// middle one of an odd number runs alone); at head_dim 128 whole q tiles of a second
// round start where the lightest of the first end.
static double small_us(const f32::PrefillPlan& p, uint32_t n_kv_heads, uint32_t head_dim,
                       uint32_t n_queries, uint32_t pos0) {
  const double t0 = head_dim == 128 ? 5.0 : 3.5, t1 = head_dim == 128 ? 4.4 : 2.5;
  const bool many = prefill_max_wg(n_kv_heads) == 1;
  auto size = [&](uint32_t qt) {
    return (uint64_t)qtile_kt(qt, p.q_per_tile, n_queries, pos0);
  };
  const uint64_t heaviest = size(p.n_qtiles - 1);
  if (p.paired) {
    const uint64_t run = heaviest + (many && p.n_qtiles == 1 ? 0 : size(0));
    uint64_t halves = 2ull * p.work_per_kvh;
    if ((many || head_dim == 128) && p.n_qtiles > 1) halves = p.n_qtiles;
    const double rounds = (double)((halves * n_kv_heads + 2 * kMaxWG - 1) / (2 * kMaxWG));
    return many && head_dim == 128 ? rounds * (t0 + t1 * run) : t0 + t1 * rounds * run;
  }
  if (head_dim == 128 && !many && p.max_splits == 1 && p.n_qtiles * n_kv_heads > kMaxWG) {
    const uint32_t last = (kMaxWG - 1) / n_kv_heads, next = kMaxWG / n_kv_heads;
    const double one = t0 + t1 * heaviest;
    const double two =
        2 * t0 + t1 * (size(p.n_qtiles - 1 - last) + size(p.n_qtiles - 1 - next));
    return one > two ? one : two;
  }
  uint64_t wg = 0, run = p.ktiles_per_split;
  for (uint32_t qt = 0; qt < p.n_qtiles; qt++) wg += (size(qt) + run - 1) / run;
  if (run > heaviest) run = heaviest;
  const double rounds = (double)((wg * n_kv_heads + kMaxWG - 1) / kMaxWG);
  return t0 + t1 * rounds * run + (p.max_splits > 1 ? 5.0 : 0.0);
}

// A kv head's q tiles either stay whole, one workgroup each (or, with more of
// them than workgroups, equal runs of them), or are cut into equal runs of key
// tiles, which costs a merge: the run with the least estimated time, from (us,
// measured) 8 + 5 per key tile of the longest run (head_dim 64: 5 + 2.8), and for
// the merge 5 + 1.3 per 8 pieces of a q tile. Calls that the f32 kernel is
// estimated to finish within 1.3 times that take it (1.1 times with more kv heads than
// half the CUs). Over 1495 drawn shapes of 1 to 128 kv heads, 8 to 2047 tokens and 0 to
// 16000 keys before them, of 10 to 150 us, both kernels timed: the one taken is 1.02
// times the better one in the mean; 61 calls are more than 3% slower than on the f32
// kernel, 24 of them more than 10%, and 94 stay on it that this one does in less than
// 0.9 of its time. A smaller margin or estimates fitted to these times trade one
// against the other. With 16 / 8 heads of 128, us, f32 kernel against this one, 64
// tokens at 2000 22.6 / 36.6, 300 at 448 27 / 33, 512 at 448 52 / 38, 300 at 2000 93 /
// 51, 200 at 16000 403 / 168.
PrefillPlan prefill_plan(uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim,
                         uint32_t n_queries, uint32_t pos0) {
  PrefillPlan p{};
  p.q_per_tile = kRows / (n_heads / n_kv_heads);
  p.n_qtiles = (n_queries + p.q_per_tile - 1) / p.q_per_tile;
  for (uint32_t qt = 0; qt < p.n_qtiles; qt++)
    p.key_tiles += qtile_kt(qt, p.q_per_tile, n_queries, pos0);
  const uint64_t most = prefill_max_wg(n_kv_heads);
  const uint64_t max_kt = qtile_kt(p.n_qtiles - 1, p.q_per_tile, n_queries, pos0);
  const uint64_t least = (p.key_tiles + most - 1) / most;
  const uint64_t rounds = (n_kv_heads + kMaxWG - 1) / kMaxWG;
  const double t0 = head_dim == 128 ? 8.0 : 5.0, t1 = head_dim == 128 ? 5.0 : 2.8;
  // Runs of whole q tiles end up to a q tile late; one run of all does not, and its
  // further q tiles cost 3 each.
  const uint64_t whole =
      p.n_qtiles <= most ? max_kt : (least > max_kt ? least : max_kt) + max_kt / 2;
  double best = most == 1 ? rounds * (t0 + 3.0 * (p.n_qtiles - 1) + t1 * p.key_tiles)
                          : t0 + t1 * rounds * whole;
  p.wg_per_kvh = (uint32_t)(p.n_qtiles < most ? p.n_qtiles : most);
  for (uint64_t run = least; run <= 4 * least && run < whole && run < p.key_tiles; run++) {
    const uint64_t pieces = (max_kt + run - 1) / run + 1;
    const double t = t0 + t1 * rounds * run + 5.0 + 1.3 * ((pieces + 7) / 8);
    if (t < best) {
      best = t;
      p.cut = true;
      p.wg_per_kvh = (uint32_t)((p.key_tiles + run - 1) / run);
    }
  }
  p.partial_slots = p.cut ? 2ull * p.wg_per_kvh * n_kv_heads : 0;
  p.small = f32::prefill_plan(n_heads, n_kv_heads, head_dim, n_queries, pos0);
  p.use_small = small_us(p.small, n_kv_heads, head_dim, n_queries, pos0) <
                (most == 1 ? 1.1 : 1.3) * best;
  return p;
}

extern "C" int32_t flock_prefill_schedule(uint32_t n_heads, uint32_t n_kv_heads,
                                          uint32_t head_dim, uint32_t n_queries, uint32_t pos0) {
  const PrefillPlan p = prefill_plan(n_heads, n_kv_heads, head_dim, n_queries, pos0);
  if (p.use_small) return 0;
  return p.cut ? 3 : p.n_qtiles == p.wg_per_kvh ? 1 : 2;
}

static uint64_t split_ws_bytes(uint64_t slots, uint32_t head_dim) {
  if (slots == 0) return 0;
  return ws_align(slots * kRows * sizeof(float2)) + slots * kRows * head_dim * sizeof(float);
}

uint64_t prefill_ws_bytes(const PrefillPlan& p, uint32_t head_dim) {
  return p.use_small ? f32::prefill_ws_bytes(p.small, head_dim)
                     : split_ws_bytes(p.partial_slots, head_dim);
}

// Upper bound over every plan with n_queries <= max_queries and pos0 +
// n_queries <= max_keys: a cut plan has at most one workgroup for each of a kv
// head's key tiles, and each of its q tiles at most those of max_keys keys. (The last
// max_queries positions need not have the most: q tiles that start elsewhere can
// end in one key tile more.)
uint64_t prefill_ws_bound(uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim,
                          uint32_t max_queries, uint32_t max_keys) {
  const uint32_t q_per_tile = kRows / (n_heads / n_kv_heads);
  const uint64_t n_qtiles = ((uint64_t)max_queries + q_per_tile - 1) / q_per_tile;
  const uint64_t key_tiles = n_qtiles * (((uint64_t)max_keys + kBK - 1) / kBK);
  const uint64_t most = prefill_max_wg(n_kv_heads);
  const uint64_t wg = key_tiles < most ? key_tiles : most;
  const uint64_t split = split_ws_bytes(wg > 1 ? 2 * wg * n_kv_heads : 0, head_dim);
  const uint64_t small =
      f32::prefill_ws_bound(n_heads, n_kv_heads, head_dim, max_queries, max_keys);
  return split > small ? split : small;
}

template <int D>
static hipError_t launch_prefill_d(const PrefillArgs& a, const PrefillTable& tab, bool cut, hipStream_t st) {
  const dim3 grid(a.n_kv_heads * a.wg_per_kvh);
  hipLaunchKernelGGL(prefill_kernel<D>, grid, dim3(kPThreads), 0, st, a, tab);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !cut) return e;
  constexpr int RPB = 256 / (D / 4);
  const dim3 mgrid(a.n_kv_heads, a.wg_per_kvh - 1, kRows / RPB);
  hipLaunchKernelGGL(prefill_merge_kernel<D>, mgrid, dim3(256), 0, st, a, tab);
  return hipGetLastError();
}

hipError_t launch_prefill(const float* q, const float* kcache, const float* vcache, float* o,
                          uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim,
                          uint32_t n_queries, uint32_t pos0, const PrefillPlan& p, void* ws,
                          hipStream_t st) {
  if (p.use_small)
    return f32::launch_prefill(q, kcache, vcache, o, n_heads, n_kv_heads, head_dim, n_queries,
                               pos0, p.small, ws, st);
  PrefillArgs a{};
  PrefillTable tab;
  a.q = q;
  a.kcache = kcache;
  a.vcache = vcache;
  a.o = o;
  if (p.cut) {
    char* w = static_cast<char*>(ws);
    a.part_ml = reinterpret_cast<float2*>(w);
    a.part_acc = reinterpret_cast<float*>(w + ws_align(p.partial_slots * kRows * sizeof(float2)));
  }
  a.n_heads = n_heads;
  a.n_kv_heads = n_kv_heads;
  a.group = n_heads / n_kv_heads;
  a.n_queries = n_queries;
  a.pos0 = pos0;
  a.q_per_tile = p.q_per_tile;
  a.n_qtiles = p.n_qtiles;
  a.wg_per_kvh = p.wg_per_kvh;
  a.scale_log2e = (float)(1.4426950408889634 / sqrt((double)head_dim));
  const bool one_each = !p.cut && p.n_qtiles == p.wg_per_kvh;
  bool pieces = false;
  uint64_t before = 0;  // key tiles before q tile `seq` of the order
  uint32_t seq = 0;
  for (uint32_t x = 0; x <= p.wg_per_kvh; x++) {
    if (one_each) {
      tab.start[x] = PrefillStart{x, 0};
      continue;
    }
    // Workgroup x starts at key tile x * key_tiles / wg_per_kvh of the order, or
    // with the q tile that holds it.
    const uint64_t at = x * p.key_tiles / p.wg_per_kvh;
    while (seq < p.n_qtiles) {
      const uint32_t n =
          qtile_kt(prefill_seq_qt(seq, p.n_qtiles), p.q_per_tile, n_queries, pos0);
      if (at < before + n) break;
      before += n;
      seq++;
    }
    tab.start[x] = PrefillStart{seq, p.cut ? (uint32_t)(at - before) : 0};
    pieces |= tab.start[x].kt != 0;
  }
  if (head_dim == 128) return launch_prefill_d<128>(a, tab, pieces, st);
  return launch_prefill_d<64>(a, tab, pieces, st);
}

}  // namespace flk
