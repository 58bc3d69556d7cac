// Attention of prompt rows over the paged cache, in one launch without partials.
//
// A decode row's keys are split over waves (attention.hip) because one token
// has no other parallelism; a prompt row has, and the split costs it: every 16
// (token, q head) pairs stream all their keys from the caches again, each
// 256-key split leaves f32 partials to merge (1.2 GB for 4,500 tokens), and one
// workgroup lists the pieces. Here a workgroup owns 128 pairs of one kv head
// (16 tokens x the 8 q heads that share it) and walks that row's keys once, so
// K and V are read once per 16 tokens and the result needs no merge: softmax,
// division and the sigmoid gate end in the same kernel.
//
// Two groups of four waves take the row's 256-key chunks in turn. Wave w of a
// group holds the q of pairs 32 w .. 32 w + 31 (64 registers) and their f32
// output tile (256 dims x 32 pairs, 128 registers); 16 KB of K and of V go from
// memory to LDS directly, one tile ahead, into two buffers per group. So a SIMD
// runs one group's softmax beside the other's products, also where a short
// prompt gives a CU only one workgroup (36 ns a key, 48 with one group), and
// the groups' halves meet once at the end. Scores are
// computed transposed, S^T = K . Q^T (v_mfma_f32_32x32x16_bf16), with the LDS
// rows of K in the order that leaves a lane with the scores of keys
// 8 h .. 8 h + 7 and 16 + 8 h .. 16 + 8 h + 7 of one pair (h its half of the
// wave): the B operand of O^T += V^T . P^T as it stands.
//
// Three prompts of 1,500 tokens (129 GFLOP with the causal half left out): 1215
// us as splits, 213 us here (0.6 PFLOP/s). What bounds it is LDS beside
// the registers: a 32-pair wave reads a tile's 32 KB for 1,024 cycles of MFMA,
// which for four SIMDs is the LDS rate; a wave of 64 pairs would halve that and
// does not fit the registers of two waves per SIMD, and with 254 of 256 in use
// only two fragment reads are under way at a time.
#include "attention.h"

#include <climits>

namespace hb {
namespace {

constexpr int kD = 256;       // head_dim
constexpr int kTile = 32;     // keys per tile
constexpr int kWaves = 4;            // waves of a key group
constexpr int kPairs = 32 * kWaves;  // (token, q head) pairs per workgroup
constexpr int kGroups = 2;           // key groups: group g takes 256-key chunks g, g + 2, ...
constexpr int kChunk = 8;            // tiles of a chunk
constexpr int kMatU4 = kTile * kD / 8;  // 16-byte units of a tile of K or of V
constexpr int kBufU4 = 2 * kMatU4;
constexpr int kBufs = 2;                // per key group
constexpr int kMergeU4 = kGroups * kWaves * 16 * 64;  // half of every wave's output tile, in the buffers' place
constexpr size_t kLds = size_t(kGroups) * kBufs * kBufU4 * 16 + kGroups * kWaves * 64 * 8;
static_assert(kMergeU4 <= kGroups * kBufs * kBufU4, "the merge fits the key buffers");
static_assert(kTile == 2 * kPage, "a tile is two pages");

typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ inline uint32_t pack_bf16x2(float lo, float hi) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, b2));
}

// v of this lane combined with v of the lane 32 further (or back)
__device__ inline float other_half_max(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__builtin_bit_cast(float, uint32_t(r[0])), __builtin_bit_cast(float, uint32_t(r[1])));
}
__device__ inline float other_half_sum(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, uint32_t(r[0])) + __builtin_bit_cast(float, uint32_t(r[1]));
}

// 64 x 16 bytes from each lane's address to LDS unit `to` onwards (lane order)
__device__ inline void to_lds(const bf16_t* from, uint4* to) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from),
                                   (__attribute__((address_space(3))) void*)(to), 16, 0, 0);
}

// Block b: q tile (last first: the longest walks start first), row, kv head.
// Rows shorter than `from` tokens are the split kernel's.
__global__ __launch_bounds__(64 * kWaves * kGroups) void attn_prefill_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache,
    const int32_t* __restrict__ block_table, int max_pages, const int32_t* __restrict__ cu_seqlens,
    const int32_t* __restrict__ context, int rows, int q_tiles, int from, int Hq, int Hkv, float scale_log2,
    const bf16_t* __restrict__ qg, int ld_qg, bf16_t* __restrict__ out) {
  extern __shared__ uint4 lds[];
  const int kh = blockIdx.x % Hkv, r = blockIdx.x / Hkv % rows, tile = q_tiles - 1 - int(blockIdx.x / Hkv / rows);
  const int lane = threadIdx.x & 63, wave8 = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int wave = wave8 % kWaves, kg = wave8 / kWaves;  // pairs 32 wave .. + 31, key group kg
  const int n32 = lane & 31, h = lane >> 5;
  const int group = Hq / Hkv;
  const int tok0 = cu_seqlens[r], T = cu_seqlens[r + 1] - tok0, ctx = context[r];
  const int pairs = T * group;
  if (!attn_prefill_row(T, ctx, from) || tile * kPairs >= pairs) return;  // uniform over the workgroup
  const int first_pos = ctx - T;                   // position of the row's first token
  // keys any pair of the workgroup sees
  const int t_last = (min(tile * kPairs + kPairs, pairs) - 1) / group;
  const int n_keys = min(first_pos + t_last + 1, ctx);
  const int n_tiles = n_keys > 0 ? (n_keys + kTile - 1) / kTile : 0;

  const int pair = tile * kPairs + wave * 32 + n32;
  const bool live = pair < pairs;
  const int t = live ? pair / group : T - 1;
  const int head = kh * group + (live ? pair % group : 0);
  const int pos = first_pos + t;  // this lane's pair sees keys 0 .. pos
  // the wave's tiles without a masked key, and with any key at all
  const int w_first = (tile * kPairs + wave * 32) / group;
  const int pos_min = first_pos + min(w_first, T - 1);
  const int pos_max = first_pos + min((tile * kPairs + wave * 32 + 31) / group, T - 1);

  // LDS row m of a K tile holds key(m): score register r of half h is then key
  // 8 h + r (r < 8) or 16 + 8 h + r - 8. Rows keep their 16-byte units XORed
  // with the row, dims of V their two halves swapped every 4 and 8 dims, so 16
  // consecutive lanes of a fragment read hit all banks; the swaps are made in
  // the addresses the lanes load from.
  const int32_t* const bt = block_table + size_t(r) * max_pages;
  const int last_page = ctx > 0 ? (ctx - 1) / kPage : 0;
  int k_src[4], v_src[4];  // element offsets within a (page, kv head) block
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = 8 * wave + 2 * i + (lane >> 5), key = 8 * ((m >> 2) & 1) + 4 * ((m >> 3) & 1) + (m & 3);
    k_src[i] = key * kD + ((lane & 31) ^ (m & 15)) * 8;
    const int u = ((4 * wave + i) * 64 + lane) & 511, d = u >> 1;
    v_src[i] = d * kPage + ((u & 1) ^ ((d >> 2) & 1) ^ ((d >> 3) & 1)) * 8;
  }
  const int my_page = wave >> 1;  // waves 0, 1 load the tile's first page, waves 2, 3 its second
  auto load_tile = [&](int i) {
    const size_t block = (size_t(bt[min(2 * i + my_page, last_page)]) * Hkv + kh) * size_t(kPage * kD);
    const bf16_t* const kp = kcache + block;
    const bf16_t* const vp = vcache + block;
    uint4* const kb = lds + (kg * kBufs + (i & 1)) * kBufU4 + wave * 256;
#pragma unroll
    for (int j = 0; j < 4; ++j) to_lds(kp + k_src[j], kb + j * 64);
#pragma unroll
    for (int j = 0; j < 4; ++j) to_lds(vp + v_src[j], kb + kMatU4 + j * 64);
  };
  if (kg * kChunk < n_tiles) load_tile(kg * kChunk);

  bf16x8 qf[16];  // B operand: dims 16 s + 8 h .. + 7 of this lane's pair
  {
    const bf16_t* const qrow = q + (size_t(tok0 + t) * Hq + head) * kD + 8 * h;
#pragma unroll
    for (int s = 0; s < 16; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qrow + 16 * s);
  }
  f32x16 o[8];
#pragma unroll
  for (int d = 0; d < 8; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[d][e] = 0.f;
  // running reference and max (base 2, the same in both halves), this half's sum
  float m = -INFINITY, row_max = -INFINITY, l = 0.f;

  const int row_u4 = n32 * 32, row_x = n32 & 15;
  const int v_u4 = n32 * 2 + (h ^ ((n32 >> 2) & 1) ^ ((n32 >> 3) & 1));
  // both groups go round equally often, group 1 past the last tile if need be
  int i = kg * kChunk;
  auto after = [](int t) { return t % kChunk == kChunk - 1 ? t + 1 + (kGroups - 1) * kChunk : t + 1; };
  for (int first = 0; first < n_tiles; first = after(first), i = after(i)) {
    // this wave's share of tile i is in LDS, then everyone's; and every wave is
    // done with the buffer the next tile goes to
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    const int next = after(i);
    if (next < n_tiles) load_tile(next);
    const int j0 = i * kTile;
    if (i >= n_tiles || j0 > pos_max) continue;  // uniform over the wave; the barriers are at the top
    const uint4* const kb = lds + (kg * kBufs + (i & 1)) * kBufU4;
    const uint4* const vb = kb + kMatU4;
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
    for (int st = 0; st < 16; ++st)
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8, kb[row_u4 + ((2 * st + h) ^ row_x)]), qf[st], s, 0, 0, 0);
    float sv[16], mx = -INFINITY;
    if (j0 + kTile - 1 <= pos_min && j0 + kTile <= ctx) {  // uniform: no masked key
#pragma unroll
      for (int e = 0; e < 16; ++e) sv[e] = s[e] * scale_log2;
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int key = j0 + (e & 8) * 2 + 8 * h + (e & 7);
        sv[e] = key <= pos && key < ctx ? s[e] * scale_log2 : -INFINITY;
      }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sv[e]);
    mx = other_half_max(mx);
    // The running max starts afresh every 256 keys, as a split of the decode
    // form does. A probability near 1 loses half as much to bf16 as one near
    // 1/2, so the reference decides the error: with one max per row the output
    // was 0.0022 - 0.0023 off the exact one instead of 0.0021 (4,500 tokens),
    // for 4 % of the time, which is what the extra rescales cost. It stays
    // within 2^16 of the row's max, so what earlier keys left cannot overflow
    // (256 keys below that weigh less than 0.4 % together).
    const bool fresh = i % kChunk == 0;
    if (__builtin_amdgcn_ballot_w64(mx > m) || fresh) {
      row_max = fmaxf(row_max, mx);
      const float m_new = fresh ? fmaxf(mx, row_max - 16.f) : fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - (m_new == -INFINITY ? 0.f : m_new));
      l *= alpha;
#pragma unroll
      for (int d = 0; d < 8; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[d][e] *= alpha;
      m = m_new;
    }
    const float ms = m == -INFINITY ? 0.f : m;
    float p[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      p[e] = __builtin_amdgcn_exp2f(sv[e] - ms);
      l += p[e];
    }
    bf16x8 pb[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const u32x4 bits = {pack_bf16x2(p[8 * k], p[8 * k + 1]), pack_bf16x2(p[8 * k + 2], p[8 * k + 3]),
                          pack_bf16x2(p[8 * k + 4], p[8 * k + 5]), pack_bf16x2(p[8 * k + 6], p[8 * k + 7])};
      pb[k] = __builtin_bit_cast(bf16x8, bits);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int d = 0; d < 8; ++d)
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vb[k * 512 + d * 64 + v_u4]), pb[k],
                                                       o[d], 0, 0, 0);
  }

  // The two key groups meet: each wave hands half of its output tile to its
  // partner (group 0 keeps dims 0 .. 127) and finishes the other half.
  f32x2* const ml = reinterpret_cast<f32x2*>(lds + kGroups * kBufs * kBufU4);  // [wave8][lane] (max, sum)
  f32x4* const swap = reinterpret_cast<f32x4*>(lds);                           // [wave8][16][lane]
  __syncthreads();  // every wave has read its last tile, and no load is under way
  ml[wave8 * 64 + lane] = f32x2{m, other_half_sum(l)};
  auto quarter = [](const f32x16& v, int e) { return f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]}; };
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x4 give = kg == 0 ? quarter(o[d + 4], 4 * e) : quarter(o[d], 4 * e);
      swap[(wave8 * 16 + d * 4 + e) * 64 + lane] = give;
    }
  __syncthreads();
  if (!live) return;  // no barrier below
  const int partner = wave8 ^ kWaves;
  const f32x2 mine = ml[wave8 * 64 + lane], other = ml[partner * 64 + lane];
  const float top = fmaxf(mine.x, other.x), ref = top == -INFINITY ? 0.f : top;
  const float wa = __builtin_amdgcn_exp2f(mine.x - ref), wb = __builtin_amdgcn_exp2f(other.x - ref);
  const float den = wa * mine.y + wb * other.y;
  const float inv = den > 0.f ? 1.f / den : 0.f;  // no visible key, or NaN scores: zeros, as the merge of the splits gives
  const bf16_t* const gate = qg + size_t(tok0 + t) * ld_qg + size_t(head) * 2 * kD + kD + kg * 128 + 4 * h;
  bf16_t* const orow = out + (size_t(tok0 + t) * Hq + head) * kD + kg * 128 + 4 * h;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int e = 0; e < 16; e += 4) {  // dims 128 kg + 32 d + 2 e + 4 h .. + 3
      const f32x4 a = kg == 0 ? quarter(o[d], e) : quarter(o[d + 4], e);
      const f32x4 b = swap[(partner * 16 + d * 4 + e / 4) * 64 + lane];
      const uint2 gv = *reinterpret_cast<const uint2*>(gate + 32 * d + 2 * e);
      const float g[4] = {__builtin_bit_cast(float, gv.x << 16), __builtin_bit_cast(float, gv.x & 0xFFFF0000u),
                          __builtin_bit_cast(float, gv.y << 16), __builtin_bit_cast(float, gv.y & 0xFFFF0000u)};
      float y[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) y[c] = (den > 0.f ? (wa * a[c] + wb * b[c]) * inv : 0.f) / (1.f + __expf(-g[c]));
      *reinterpret_cast<uint2*>(orow + 32 * d + 2 * e) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
    }
}

}  // namespace

bool attn_prefill_rows(const AttnGeom& g, AttnWork& w, int tokens, const bf16_t* qg, int ld_qg, const bf16_t* out) {
  auto aligned = [](const void* p, uintptr_t n) { return reinterpret_cast<uintptr_t>(p) % n == 0; };
  w.prefill_from = 0;
  w.prefill_only = false;
  if (w.max_tokens < kPrefillRowTokens || g.head_dim != kD || ld_qg % 4 != 0 || !aligned(qg, 8) || !aligned(out, 8))
    return false;
  const int64_t pairs = int64_t(w.max_tokens) * (g.q_heads / g.kv_heads);
  if (pairs > INT_MAX / 2 || (pairs + kPairs - 1) / kPairs * w.rows * g.kv_heads > INT_MAX) return false;
  w.prefill_from = kPrefillRowTokens;
  // the other rows hold at most max_tokens each: the shortest has at least the rest
  const int64_t least = int64_t(tokens) - int64_t(w.rows - 1) * w.max_tokens;
  w.prefill_only = attn_prefill_row(least, int64_t(w.splits) * w.split_len, w.prefill_from);
  return true;
}

void attn_prefill(const bf16_t* q, const bf16_t* kcache, const bf16_t* vcache, const int32_t* block_table,
                  int max_pages, const int32_t* cu_seqlens, const int32_t* context, const AttnGeom& g, float scale,
                  const AttnWork& w, const bf16_t* qg, int ld_qg, bf16_t* out, hipStream_t stream) {
  require(w.prefill_from > 0, "attn_prefill: no rows for it");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(attn_prefill_kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(kLds));
  HB_CHECK(attr);
  const int q_tiles = (w.max_tokens * (g.q_heads / g.kv_heads) + kPairs - 1) / kPairs;
  launch_timed(attn_prefill_kernel, dim3(unsigned(q_tiles) * w.rows * g.kv_heads), dim3(64 * kWaves * kGroups), kLds, stream, q,
               kcache, vcache, block_table, max_pages, cu_seqlens, context, w.rows, q_tiles, w.prefill_from, g.q_heads,
               g.kv_heads, scale * 1.44269504088896340736f, qg, ld_qg, out);
  HB_CHECK(hipGetLastError());
}

}  // namespace hb
