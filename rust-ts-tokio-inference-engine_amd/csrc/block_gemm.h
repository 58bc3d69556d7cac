// 4-bit projections and expert products of prompt-sized steps: y = x . W^T,
// W = s*q + b per group of 64, tiled layout of q4_tile. Device template:
// included by qmm.hip (dense) and moe.hip (grouped).
//
// Workgroup: 4 waves, 256 weight rows x up to 96 tokens; wave w owns rows
// 64 w .. 64 w + 63 over the whole K and every token of the block (two 32-row by
// three 32-token tiles of v_mfma_f32_32x32x16_bf16, 96 accumulators). What a
// decode-sized kernel spends per output (dequantising a fragment, reading x
// from LDS) falls with the tile: a fragment is dequantised once for 96 tokens
// and an LDS read of x serves 64 weight rows, where the 16-row wave of the
// streaming kernel reads LDS for twice as long as its matrix instructions take.
// What is left beside the matrix work is mostly the f32 scaling, one FMA per
// output and group; all vector work is put between matrix instructions, and two
// workgroups share a CU (250 of 256 registers). 128 tokens a wave need 33
// vector registers more than that leaves for the interleaving and took the same
// time.
//
// x goes from memory to LDS directly, one 64-column group a stage, two stages
// ahead in a ring of three; a wave's weights take the same way a pair of groups
// ahead (its own 4 KB, read by it alone), so that nothing in flight holds
// registers.
//
// Measured (us, streaming kernel before / here): 2,000 tokens x [12544, 2048]
// 242 / 140 (0.73 PFLOP/s), 4,000 473 / 268; 4,000 x [2048, 4096] 271 / 126.
// Bound by the vector pipe and the waits between stages: matrix instructions
// fill 34 % of the cycles, vector ones 46 %.
//
// Arithmetic: total += s * (sum x (16 + q)) per group in f32, and the rest, sum
// over groups of (b - 16 s) * (sum of x over the group), as bf16 products: the
// group sums in three bf16 parts (24 bits), b and -16 s exact in bf16. That is
// 12 matrix instructions per 16 groups and tile instead of 32 slower f32 ones,
// and every product is exact. The offset 16 is the smallest whose sixteen codes
// share an exponent (0x4180 | q << 3), for one more shift per word than 128:
// the f32 sums it is taken out of again stay eight times smaller.
#pragma once
#include "hb_common.h"
#include "q4_device.h"

namespace hb {
namespace {

constexpr int kBgWaves = 4;
constexpr int kBgThreads = 64 * kBgWaves;
constexpr int kBgRows = 64 * kBgWaves;  // weight rows per workgroup
constexpr int kBgTok = 96;              // tokens per workgroup
constexpr int kBgTokWave = kBgTok / kBgWaves;  // that a wave stages and sums
constexpr int kBgRing = 3;              // x stages in LDS
constexpr int kBgStageU4 = kBgTok * 8;  // uint4 of a stage: 64 columns of every token
constexpr int kBgSumGroups = 16;        // groups between bias products
constexpr int kBgSumLd = 20;            // floats per token of the group sums
constexpr int kBgWeightU4 = kBgRows / 16 * 64;  // uint4 of a pair of groups of the block's weights
constexpr size_t kBgLds = size_t(kBgRing * kBgStageU4 + 2 * kBgWeightU4) * 16 + size_t(kBgTok) * kBgSumLd * 4;
static_assert(2 * kBgLds <= 160 * 1024, "two workgroups per CU");

__device__ inline f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// bf16 (16 + code) for the 8 codes of one interleaved word, in k order: as
// q4_offset_bf16_s, with the codes three bits higher
__device__ inline Q4Consts bg_consts() {
  Q4Consts c{0x00780078u, 0x41804180u};
  asm volatile("" : "+v"(c.mask), "+s"(c.magic));
  return c;
}
__device__ inline bf16x8 bg_offset16(uint32_t w, Q4Consts c) {
  u32x4 d;
  d[0] = and_or_b32(w << 3, c.mask, c.magic);
  d[1] = and_or_b32(w >> 1, c.mask, c.magic);
  d[2] = and_or_b32(w >> 5, c.mask, c.magic);
  d[3] = and_or_b32(w >> 9, c.mask, c.magic);
  return __builtin_bit_cast(bf16x8, d);
}

// Three bf16 parts of eight f32 values (hi + mid + lo is the value to 2^-24 of it)
__device__ inline void split3(const float (&f)[8], bf16x8 (&part)[3]) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  u32x4 bits[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = f[2 * i], b = f[2 * i + 1];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, b2));
      bits[p][i] = u;
      a -= __builtin_bit_cast(float, u << 16);
      b -= __builtin_bit_cast(float, u & 0xFFFF0000u);
    }
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) part[p] = __builtin_bit_cast(bf16x8, bits[p]);
}

// Sum of a unit's eight bf16 values in f32
__device__ inline float bg_unit_sum(u32x4 v) {
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const b2 one = __builtin_bit_cast(b2, 0x3F803F80u);
  float s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, uint32_t(v[0])), one, 0.f, false);
  s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, uint32_t(v[1])), one, s, false);
  s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, uint32_t(v[2])), one, s, false);
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, uint32_t(v[3])), one, s, false);
}

// Workgroup barrier for LDS, without the fences at which the compiler waits for
// every load to LDS under way: this wave's own LDS operations are done, and the
// compiler moves none across
__device__ inline void bg_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// Keeps this wave's LDS reads behind its own loads to LDS (waited for before it)
__device__ inline void wave_lds_order() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local"); }

// What a block multiplies: `rows` live tokens (1..128) at x + xrow[..] K-wide
// rows, weight tiles from `tile` on (16 rows each), both over PK = K / 128 pairs.
struct BgBlock {
  const bf16_t* x;  // uniform base
  int rows;
  const uint4* w;   // first 16-row tile of the block's weights
  const uint2* sb;
};

// total[t][j][r]: token 32 t + 8 (r >> 2) + 4 h + (r & 3), weight row
// 64 wave + 32 j + (lane & 31). TT: 32-token tiles computed. xoff: this lane's
// byte offsets of the four token rows it stages (token 32 wave + 8 i +
// lane / 8, with the 16-byte unit it reads of each 64-column group).
template <int TT>
__device__ inline void bg_run(const BgBlock& blk, const uint32_t (&xoff)[kBgTokWave / 8], int PK, uint4* lds, f32x16 (&total)[TT][2]) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int n32 = lane & 31, h = lane >> 5;
  uint4* const wl = lds + kBgRing * kBgStageU4 + wave * 256;  // this wave's four 16-row tiles of a pair, two buffers
  float* const sums = reinterpret_cast<float*>(lds + kBgRing * kBgStageU4 + 2 * kBgWeightU4);  // [token][kBgSumLd]
  const Q4Consts magic = bg_consts();
  const int groups = 2 * PK;

  auto load_x = [&](int g, int slot) {  // 64 columns of the block's tokens, past the last group that one again
    const char* const xg = reinterpret_cast<const char*>(blk.x + size_t(min(g, groups - 1)) * 64);
    uint4* const to = lds + slot * kBgStageU4 + wave * kBgTokWave * 8;
#pragma unroll
    for (int i = 0; i < kBgTokWave / 8; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xg + xoff[i]),
                                       (__attribute__((address_space(3))) void*)(to + i * 64), 16, 0, 0);
  };
  // lane (n, h) of 32-row tile j takes the words of quarters 2 h and 2 h + 1 of
  // its row: codes 16 (2 h + a) .. + 15 of each group, a = 0, 1
  const uint4* const wg = blk.w + size_t(4 * wave) * PK * 64 + lane;
  const int wread = (n32 >> 4) * 64 + 32 * h + (lane & 15);
  const uint2* const sp = blk.sb + size_t(4 * wave + (n32 >> 4)) * PK * 16 + (lane & 15);
  uint2 sbr[2];
  float psc[2][2];  // [group of the pair][32-row tile] scales
  auto scales = [&] {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      psc[0][j] = __builtin_bit_cast(float, sbr[j].x << 16);
      psc[1][j] = __builtin_bit_cast(float, sbr[j].y << 16);
      asm volatile("" : "+v"(psc[0][j]), "+v"(psc[1][j]));  // here, before newer loads are out
    }
  };
  auto load_w = [&](int p) {
    const int pc = min(p, PK - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wg + (size_t(i) * PK + pc) * 64),
                                       (__attribute__((address_space(3))) void*)(wl + (p & 1) * kBgWeightU4 + i * 64), 16, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) sbr[j] = sp[(size_t(2 * j) * PK + pc) * 16];
  };
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) total[t][j][r] = 0.f;
  f32x16 zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.f;

  // this lane's words of row tile j, both groups of the pair. Every read of the
  // buffers is a bit cast of a whole uint4 (kept whole by the asm below): before
  // copied or merged ones the compiler waits for all loads to LDS under way.
  auto read_words = [&](int p, int j, u32x4 (&v)[2]) {
#pragma unroll
    for (int a = 0; a < 2; ++a) v[a] = __builtin_bit_cast(u32x4, wl[(p & 1) * kBgWeightU4 + 128 * j + wread + 16 * a]);
  };
  auto dequant = [&](u32x4 (&v)[2], int gi, bf16x8 (&w)[4]) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      asm("" : "+v"(v[a]));
      w[2 * a] = bg_offset16(v[a][2 * gi], magic);
      w[2 * a + 1] = bg_offset16(v[a][2 * gi + 1], magic);
    }
  };
  load_w(0);
  load_x(0, 0);
  load_x(1, 1);
  const int xr = n32 * 8, xs = (n32 >> 1) & 7;  // fragment row and swizzle of token n32 (tokens 32 t + n32 alike)
  bf16x8 wf[2][4];
  {
    u32x4 v[2];
    __builtin_amdgcn_s_waitcnt(0x0f76);  // vmcnt(6): all but the two x stages
    wave_lds_order();
    read_words(0, 0, v);
    dequant(v, 0, wf[0]);
    scales();
  }

  int slot = 0;
  for (int p = 0; p < PK; ++p) {
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
      const int g = 2 * p + gi;
      // Stage g of x has arrived, for every wave, and every wave is done with
      // the buffer stage g + 2 goes to. Loads to LDS end in order: stage g's were
      // issued two stages ago, and after them the next stage's three and, between
      // a pair's two stages, the next pair's weights (four, not counting the
      // scales, which go to registers).
      if (gi == 0)
        __builtin_amdgcn_s_waitcnt(0x0f73);  // vmcnt(3)
      else
        __builtin_amdgcn_s_waitcnt(0x0f77);  // vmcnt(7)
      bg_barrier();
      const float sc[2] = {psc[gi][0], psc[gi][1]};
      if (gi == 0) load_w(p + 1);
      __builtin_amdgcn_sched_barrier(0);
      load_x(g + 2, slot == 0 ? 2 : slot - 1);
      const uint4* const xb = lds + slot * kBgStageU4;
      slot = slot == 2 ? 0 : slot + 1;
      auto frag = [&](int t, int u) { return __builtin_bit_cast(bf16x8, xb[t * 256 + xr + ((4 * h + u) ^ xs)]); };
      bf16x8 f[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) f[u] = frag(0, u);
      u32x4 words[2];
      read_words(p, 1, words);
      // two of the four units of token st that this lane sums, addresses derived
      // here (kept, they cost the registers that the tiles need)
      int ln = lane;
      asm volatile("" : "+v"(ln));
      auto units = [&](int i, u32x4 (&v)[2]) {
        const int tok = kBgTokWave * wave + min(ln >> 1, kBgTokWave - 1);
#pragma unroll
        for (int k = 0; k < 2; ++k) v[k] = __builtin_bit_cast(u32x4, xb[tok * 8 + ((4 * (ln & 1) + i + k) ^ ((tok >> 1) & 7))]);
      };
      u32x4 sv[2];
      units(0, sv);
      float unit_sum = 0.f;
      auto first_sum = [&] {
        unit_sum = bg_unit_sum(sv[0]) + bg_unit_sum(sv[1]);
        units(2, sv);
      };
      auto second_sum = [&] {
        float v = unit_sum + (bg_unit_sum(sv[0]) + bg_unit_sum(sv[1]));
        v += __builtin_bit_cast(float,
                                __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
        sums[(kBgTokWave * wave + min(ln >> 1, kBgTokWave - 1)) * kBgSumLd + g % kBgSumGroups] = v;  // both lanes the same
      };
      __builtin_amdgcn_sched_barrier(0);
      // (token tile, row tile) steps in turn. What the vector pipe has to do goes
      // between the matrix instructions: the scaling of the step before, the
      // second row tile's codes and the group sums in the first steps, the first
      // row tile's codes of the next stage in the last; and a fragment of the
      // next token tile is read as soon as the last product with this one's is out
      f32x16 acc[2];
      auto scale = [&](int t, int j) {
#pragma unroll
        for (int r = 0; r < 16; ++r) total[t][j][r] = __builtin_fmaf(sc[j], acc[j][r], total[t][j][r]);
        asm volatile("" : "+v"(total[t][j]));  // here, not where the compiler would sink it to
      };
#pragma unroll
      for (int t = 0; t < TT; ++t) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const bool first = t == 0 && j == 0, second = t == 0 && j == 1;
          const bool last = t == TT - 1 && j == 1;
          if (last) {
            if (gi == 1) {
              __builtin_amdgcn_s_waitcnt(0x0f76);  // vmcnt(6): the next pair's words, before two x stages
              wave_lds_order();
            }
            read_words(p + gi, 0, words);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            acc[j] = mfma32(f[u], wf[j][u], u ? acc[j] : zero);
            if (j == 1 && t + 1 < TT) f[u] = frag(t + 1, u);
          }
          if (j == 1)
            scale(t, 0);
          else if (t > 0)
            scale(t - 1, 1);
          if (first) {
            dequant(words, gi, wf[1]);
            first_sum();
          }
          if (second) second_sum();
          if (last) dequant(words, gi ^ 1, wf[0]);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                            // one matrix instruction
            if (j == 1 && t + 1 < TT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
            if (first || second)  // vector instructions
              __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
            else if (last)
              __builtin_amdgcn_sched_group_barrier(0x002, 12, 0);
            else
              __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      scale(TT - 1, 1);
      if (gi == 1) scales();
    }
    // the bias products of the last groups (a multiple of 16, or the rest of K)
    if ((2 * p + 2) % kBgSumGroups == 0 || p == PK - 1) {
      const int g0 = (2 * p + 1) / kBgSumGroups * kBgSumGroups;
      bf16x8 bb[2], bs[2];  // b and -16 s of groups g0 + 8 h .. + 7 of this lane's rows
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        u32x4 vb, vs;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int q = g0 / 2 + 4 * h + i;  // pair
          uint2 v = sp[(size_t(2 * j) * PK + min(q, PK - 1)) * 16];
          if (q >= PK) v = uint2{0u, 0u};
          vb[i] = (v.x >> 16) | (v.y & 0xFFFF0000u);
          vs[i] = (__builtin_bit_cast(uint32_t, -16.f * __builtin_bit_cast(float, v.x << 16)) >> 16) |
                  (__builtin_bit_cast(uint32_t, -16.f * __builtin_bit_cast(float, v.y << 16)) & 0xFFFF0000u);
        }
        bb[j] = __builtin_bit_cast(bf16x8, vb);
        bs[j] = __builtin_bit_cast(bf16x8, vs);
      }
      bg_barrier();  // every token's sums are written; the next stage's barrier ends their reading
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        float f[8];
        const f32x4* const row = reinterpret_cast<const f32x4*>(sums + (32 * t + n32) * kBgSumLd + 8 * h);
        const f32x4 lo = row[0], hi = row[1];
        const int have = groups - g0 - 8 * h;  // groups of this half that exist
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f[i] = i < have ? lo[i] : 0.f;
          f[i + 4] = i + 4 < have ? hi[i] : 0.f;
        }
        bf16x8 part[3];
        split3(f, part);
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            total[t][j] = mfma32(part[q], bb[j], total[t][j]);
            total[t][j] = mfma32(part[q], bs[j], total[t][j]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the repeated last loads may not outlive the workgroup's LDS
}

// two floats to a bf16 pair, round to nearest even
__device__ inline uint32_t bg_pack(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo, hi}, b2));
}

// Blocks of a dense matrix: block b on XCD b % 8, j = b / 8: token block
// j % tblocks, row block (j / tblocks) * 8 + b % 8, so the token blocks of a row
// block run side by side on one XCD and its weights come from HBM once.
// OUT 0: y bf16, 1: y f32, 2: y f32 +=.
template <int OUT, int TT>
__device__ inline void bg_dense(const BgBlock& blk, const uint32_t (&xoff)[kBgTokWave / 8], int PK, uint4* lds, void* yv, int ldy,
                                size_t m0, int row0) {
  f32x16 total[TT][2];
  bg_run<TT>(blk, xoff, PK, lds, total);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = row0 + 64 * wave + 32 * j + n32;
      if constexpr (OUT == 0) {
        // two columns per store: the even lane of a pair takes the even tokens
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          float even = total[t][j][r], odd = total[t][j][r + 1];
          asm("" : "+v"(even), "+v"(odd));  // two registers to choose from, not an index into sixteen
          const float give = (lane & 1) ? even : odd, keep = (lane & 1) ? odd : even;
          const float got = __builtin_bit_cast(
              float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, give), 0xB1, 0xF, 0xF, false));
          const int m = 32 * t + 8 * (r >> 2) + 4 * h + (r & 3) + (lane & 1);
          const uint32_t pair = (lane & 1) ? bg_pack(got, keep) : bg_pack(keep, got);
          if (m < blk.rows)
            *reinterpret_cast<uint32_t*>(static_cast<bf16_t*>(yv) + (m0 + m) * ldy + (col & ~1)) = pair;
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
          if (m >= blk.rows) continue;
          float* const y = static_cast<float*>(yv) + (m0 + m) * ldy + col;
          *y = OUT == 2 ? *y + total[t][j][r] : total[t][j][r];
        }
      }
    }
}

template <int OUT>
__global__ __launch_bounds__(kBgThreads, 2) void block_gemm_kernel(const bf16_t* __restrict__ x, int M, int PK,
                                                                 const uint32_t* __restrict__ wt,
                                                                 const bf16_t* __restrict__ sbt, int n_rows,
                                                                 int tblocks, void* __restrict__ yv, int ldy) {
  extern __shared__ uint4 lds[];
  const int b = blockIdx.x, j8 = b / 8;
  const int tb = j8 % tblocks, rb = (j8 / tblocks) * 8 + b % 8;
  if (rb >= n_rows / kBgRows) return;  // uniform over the workgroup
  const size_t m0 = size_t(tb) * kBgTok;
  const int K = PK * 128, rows = min(kBgTok, M - int(m0));
  BgBlock blk{x + m0 * K, rows, reinterpret_cast<const uint4*>(wt) + size_t(rb) * (kBgRows / 16) * PK * 64,
              reinterpret_cast<const uint2*>(sbt) + size_t(rb) * (kBgRows / 16) * PK * 16};
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t xoff[kBgTokWave / 8];
#pragma unroll
  for (int i = 0; i < kBgTokWave / 8; ++i) {
    const int t = kBgTokWave * wave + 8 * i + (lane >> 3);
    xoff[i] = uint32_t(min(t, rows - 1)) * uint32_t(K) * 2u + ((lane & 7) ^ ((t >> 1) & 7)) * 16;
  }
  if (rows > 64)
    bg_dense<OUT, 3>(blk, xoff, PK, lds, yv, ldy, m0, rb * kBgRows);
  else
    bg_dense<OUT, 2>(blk, xoff, PK, lds, yv, ldy, m0, rb * kBgRows);
}

// Runs the block form for M > kBgMinTokens when the shape and the operands'
// alignment suit it and there are blocks enough; false otherwise, nothing
// launched. Up to 256 tokens (decode and verify steps) a row's bits may not
// depend on the batch, so those keep the kernels whose sums have one order.
// Blocks: a lone one takes 40 us at K = 2048 however many there are beside it,
// up to two per CU (us before / here: 300 x [12544, 2048] = 196 blocks 44 / 40,
// 2,000 x [2048, 4096] = 168 144 / 96; 4,000 x [768, 2048] = 126 59 / 57,
// 1,000 x [2048, 4096] = 88 77 / 94).
constexpr int kBgMinTokens = 256, kBgMinBlocks = 160;

template <int OUT>
bool block_gemm(const bf16_t* x, int M, int K, const uint32_t* w, const bf16_t* sb, int n_rows, void* y, int ldy,
                hipStream_t stream) {
  // a longer K is taken, or refused, by the other forms alone
  if (M <= kBgMinTokens || n_rows % kBgRows || K % 128 || K > 4096) return false;
  if (OUT == 0 && (ldy % 2 || reinterpret_cast<uintptr_t>(y) % 4)) return false;
  const int rblocks = n_rows / kBgRows, tblocks = (M + kBgTok - 1) / kBgTok;
  const int64_t blocks = int64_t((rblocks + 7) / 8 * 8) * tblocks;
  if (int64_t(rblocks) * tblocks < kBgMinBlocks) return false;
  if (blocks > 0x7FFFFFFF || int64_t(K) * 2 * kBgTok > 0x7FFFFFFF) return false;
  const auto kernel = &block_gemm_kernel<OUT>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(kBgLds));
  HB_CHECK(attr);
  hipLaunchKernelGGL(kernel, dim3(unsigned(blocks)), dim3(kBgThreads), kBgLds, stream, x, M, K / 128, w, sb, n_rows,
                     tblocks, y, ldy);
  return true;
}

}  // namespace
}  // namespace hb
