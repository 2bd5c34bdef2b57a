// Matrix products whose row tiles are tall: an expert's rows times its weights where an expert sees dozens of rows or more, and
// plain linears of prefill chunks (with SiLU and the product with the up projection, or cut along K).  y = x W^T in the swapped form of skinny_gemm.hip, D = W . x^T, on the same
// LDS image of 128-byte rows (16-byte chunk c of row r at c ^ ((r >> 1) & 7): conflict-free for 32-row fragments as well).
//
// What bounds it: the matrix cores, and through them the power limit (at 90 % of busy matrix cores the chip runs at 1.37 GHz).
//   * A tile is 256 rows x 256 weight rows, a wave's part 128 x 128: 1 KiB of LDS reads per two 32x32x16 products.  Eight waves of
//     128 x 32, the ring kernel's split, read 160 KB of LDS per 64-wide k block for half the products, more than its port delivers.
//   * Four waves, one per SIMD, no loader waves: fragments of the next half k block are read while the current ones are multiplied,
//     with the compiler's own waits.  The two stages are static LDS objects of their own: hipcc then knows that a load into one
//     does not touch the other (a single array would drain every load in flight in front of each fragment read).
//   * 32x32x16 products: their accumulators are updated in place.  With 16x16x32 the compiler rotates 256 registers through copies.
//   * Loads are spread over the step, one per two or three products: a burst of sixteen fills the memory pipe's queue, and a wave
//     that waits for a place in it issues no products either (16 in a row 0.96, spread 1.42 PFLOP/s at 65536 x 8192 x 4096).
//   * A workgroup stays and takes its XCD's items in turn; the next item's first two stages are on their way through the last two
//     steps, and its places are fetched a whole item ahead.  Results turn in LDS and leave as 256-byte row segments.
//   * Experts' weight rows a multiple of 4096 bytes apart: the k blocks of a tile begin where those of the other grouped kernels do
//     (skinny_grouped.h; one order of sums).  Up, relu squared, 4096 x 1536, 1000 tokens, 8 chosen 191 | 186 us, gated, 6 chosen 313 | 294, 2048
//     x 768, 1000 tokens 57 | 50; from 2048 tokens on 0.99 to 1.01 of the time without.
//   * A row tile's live rows are counted in units of 64: four code paths, so that an expert's last tile costs what it holds.
// Experts' both products, 4096 x 1536, 64 experts, 8 chosen (relu squared): 8192 rows 2176 -> 1603 us, 1024 rows 877 -> 400 us;
// gated, 6 chosen: 8192 rows 2289 -> 1819 us, 1365 rows 1213 -> 533 us; 1024 x 384, 128 experts, 8 chosen: 2048 rows 199 -> 113 us
// (before: the ring kernel's 64- and 256-row tiles).  Linears beside the library's: layers.py, _tall_wins.
#include "mfma_attn_common.h"
#include "skinny_grouped.h"
#include "skinny_tile.h"

namespace mi {
namespace {

struct TallParams {
  const uint16_t* x;
  const uint16_t* w;
  uint16_t* out;
  int32_t N, K;
  int32_t rpt, gather_div;      // rows per tile; > 0: source row = pair index / gather_div, else the row itself
  int32_t nx;                   // weight tiles
  uint32_t div_magic;           // 2^32 / gather_div, rounded up: exact for pair indices below 2^28
  const int32_t* row_map;       // [max_rows] pair index or -1
  const int32_t* tile_expert;   // [max_tiles]
  const int32_t* num_tiles;     // [1]
  const float* pair_weights;    // RELU_SQUARED: the sums of a pair's row times this, in front of the activation
  int64_t ldx, ldo, w_expert_stride;
  int32_t turn;      // the TURN form: experts whose tiles' k blocks begin with grouped_first_block and go round
  // DENSE: one weight matrix, all M rows.  The first `whole` tiles are items of their own; each of the others is cut along K into
  // `split` items that leave fp32 sums in part [item][256][256]
  int32_t M, whole, split, group;
  const uint16_t* bias;
  float* part;
};

// FORM of a dense product (the others are MI_MOE_*)
constexpr int kTallDense = 16, kTallDenseGated = 17;
constexpr bool tall_dense(int form) { return form >= kTallDense; }
constexpr bool tall_gated(int form) { return form == MI_MOE_GATED || form == kTallDenseGated; }

constexpr int kTallN = 256;       // weight rows of a tile
constexpr int kTallStage = 64 * 1024;

// the part of a work item that its place decides; row: the item's 8 x pieces' rows of a_rows, as the alignment's map has them
struct TallItem {
  int row0, tile, expert, units;     // units: 64-row units of the row tile that hold live rows
  int kb, n_it;                      // where the item starts along K (bytes) and its 64-wide blocks: an even number
  int first;                         // TURN: the block that it begins with (then round)
  int slab;                          // >= 0: fp32 sums into this slab
  int row[8];
};

// items of the XCD-th of eight workgroup sets: a range of the whole tiles, then a range of the pieces
__device__ __forceinline__ int tall_items(const TallParams& p, bool dense, int xcd, int& lo, int& whole, int& tail) {
  const int work = dense ? p.whole : p.num_tiles[0] * p.nx, each = (work + 7) >> 3;
  lo = xcd * each;
  whole = max(min(each, work - lo), 0);
  tail = 0;
  if (dense && p.split > 1) {
    const int pieces = (((p.M + 255) >> 8) * p.nx - p.whole) * p.split, per = (pieces + 7) >> 3;
    tail = xcd * per;
    return whole + max(min(per, pieces - tail), 0);
  }
  return whole;
}

template <int FORM, bool TURN>
__device__ __forceinline__ void tall_fetch(const TallParams& p, int item, int lo, int whole, int tail, TallItem& t) {
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  t.kb = 0;
  t.n_it = p.K >> 6;
  t.slab = -1;
  if constexpr (tall_dense(FORM)) {
    int at = lo + item;
    if (item >= whole) {
      t.slab = tail + item - whole;
      const int s = t.slab % p.split, nb = p.K >> 7, b0 = s * nb / p.split;
      at = p.whole + t.slab / p.split;
      t.kb = b0 * 256;
      t.n_it = 2 * ((s + 1) * nb / p.split - b0);
    }
    // `group` row tiles by the weight tiles, rows first: what an XCD's 32 workgroups read at a time
    const int tiles = (p.M + 255) >> 8, g = at / (p.group * p.nx), in = at - g * p.group * p.nx, rows = min(p.group, tiles - p.group * g);
    t.tile = in / rows;
    t.row0 = (p.group * g + in - t.tile * rows) * 256;
    t.units = min((p.M - t.row0 + 63) >> 6, 4);
    t.expert = 0;
    return;
  }
  item += lo;
  const int row_tile = item / p.nx;      // the weight tiles of a row tile in a row: its rows through one L2
  t.tile = item - row_tile * p.nx;
  t.row0 = row_tile * p.rpt;
  t.expert = p.tile_expert[row_tile];
  if constexpr (TURN) t.first = grouped_first_block(tall_gated(FORM), t.expert, t.tile * (tall_gated(FORM) ? kTallN / 2 : kTallN), p.N, t.n_it);
  t.units = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (u < p.rpt / 64 && __ballot(p.row_map[t.row0 + 64 * u + lane] >= 0)) t.units = u + 1;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 8 * (wid + 4 * i) + (lane >> 3);
    const int r = t.row0 + (row < p.rpt ? row : 0);
    t.row[i] = p.gather_div > 0 ? p.row_map[r] : r;
  }
}

// where block i of an item lies along K (bytes)
template <bool TURN>
__device__ __forceinline__ int tall_block(const TallItem& t, int i) {
  if constexpr (!TURN) return t.kb + i * 128;
  const int at = i + t.first;
  return (at < t.n_it ? at : at - t.n_it) * 128;
}

// byte offsets of a lane's 8 x pieces
template <int FORM>
__device__ __forceinline__ void tall_rows(const TallParams& p, const TallItem& t, uint32_t (&x)[8]) {
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 8 * (wid + 4 * i) + (lane >> 3);
    const int lc = (lane & 7) ^ ((row >> 1) & 7);
    if constexpr (tall_dense(FORM)) {     // a row past the last one repeats it and is never stored
      x[i] = (uint32_t)min(t.row0 + row, p.M - 1) * (uint32_t)(2 * p.ldx) + 16 * lc;
      continue;
    }
    uint32_t m = t.row[i] < 0 ? 0u : (uint32_t)t.row[i];
    if (p.gather_div > 1) m = __umulhi(m, p.div_magic);      // / gather_div
    x[i] = m * (uint32_t)(2 * p.ldx) + 16 * lc;
  }
}

template <bool GATED>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tall_weights(const TallParams& p, const TallItem& t) {
  // what hangs over an expert's last row reads as zero and is never stored
  const int64_t first = (int64_t)t.tile * (GATED ? kTallN / 2 : kTallN) * p.K;
  const int64_t all = (int64_t)(GATED ? 2 : 1) * p.N * p.K;
  return __builtin_amdgcn_make_buffer_rsrc((void*)(p.w + (int64_t)t.expert * p.w_expert_stride + first), 0, (int)(uint32_t)((all - first) * 2), 0x00020000);
}

// wo: byte offsets of a lane's 8 weight pieces
__device__ __forceinline__ void tall_issue_w(const uint32_t (&wo)[8], __amdgpu_buffer_rsrc_t wr, int kb, char* st) {
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(st + (wid + 4 * i) * 1024), 16, wo[i], kb, 0, 0);
}
// XP: pieces of x a wave loads (2 per 64-row unit)
template <int XP>
__device__ __forceinline__ void tall_issue_x(const TallParams& p, const uint32_t (&x)[8], int kb, char* st) {
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, -1, 0x00020000);
#pragma unroll
  for (int i = 0; i < XP; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(st + 32768 + (wid + 4 * i) * 1024), 16, x[i], kb, 0, 0);
}

constexpr int vmcnt_imm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
constexpr int kLgkm0 = 0xC07F;     // lgkmcnt(0), any vmcnt

// A tile of 64 HM rows x 256 weight rows.  Four waves: 2 (rows) x 2 (weight rows), each 32 HM x 128.
template <typename Tag, int FORM, bool TURN, int HM>
__device__ __forceinline__ void tall_tile(const TallParams& p, char* s0, char* s1, char* so, const TallItem& t, uint32_t (&x)[8],
                                          const uint32_t (&wo)[8], const TallItem& nt, bool more) {
  using E = Elem<Tag>;
  constexpr bool GATED = tall_gated(FORM);
  constexpr int NM = 8 * HM;                 // products of half a step
  constexpr int PPL = 8 + 2 * HM;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid & 1, wn = wid >> 1;
  const int n_it = t.n_it;
  const int r32 = lane & 31, half = lane >> 5;
  int frag[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) frag[k] = r32 * 128 + ((((k & 1 ? 2 + 2 * half : 6 * half) + (k >> 1)) ^ ((r32 >> 1) & 7)) << 4);
  const int x_off = 32768 + wm * (HM * 4096), w_off = wn * 16384;
  f32x16_t acc[4][HM];
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int j = 0; j < HM; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[g][j][i] = 0.f;
  uint4 a[2][2][4], b[2][2][HM];
  auto read = [&](int u, const char* st) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        a[u][k][g] = __builtin_bit_cast(uint4, *reinterpret_cast<const u32x4_t*>(st + frag[2 * u + k] + w_off + g * 4096));
#pragma unroll
      for (int j = 0; j < HM; ++j)
        b[u][k][j] = __builtin_bit_cast(uint4, *reinterpret_cast<const u32x4_t*>(st + frag[2 * u + k] + x_off + j * 4096));
    }
  };
  auto mul = [&](int u, int lo, int hi) __attribute__((always_inline)) {
#pragma unroll
    for (int i = lo; i < hi; ++i) {
      const int k = i / (4 * HM), g = i % 4, j = i % (4 * HM) / 4;
      acc[g][j] = mfma32<Tag>(a[u][k][g], b[u][k][j], acc[g][j]);
    }
  };
  __amdgpu_buffer_rsrc_t wr = tall_weights<GATED>(p, t);
  auto barrier = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int A = NM * 5 / 8, B = NM / 4;      // where the two barriers of a step stand among its 2 NM products
  int ahead = TURN ? tall_block<TURN>(t, 2) : 0;      // where the next step's loads lie along K
  // KIND 0: a step in the middle; 1, 2: the last two, which load the next item's first two
  auto step = [&](auto kind, int it, char* cur, char* nxt) __attribute__((always_inline)) {
    constexpr int KIND = decltype(kind)::value;
    int kb = KIND == 0 ? t.kb + (it + 2) * 128 : tall_block<TURN>(nt, KIND - 1);
    if constexpr (TURN && KIND == 0) {
      // (here, among the products: behind the barrier, in front of the loads, it costs 1 to 2 % of a launch that the matrix cores hold)
      kb = ahead;
      ahead = ahead + 128 == 128 * n_it ? 0 : ahead + 128;
      asm volatile("" : "+s"(kb), "+s"(ahead));
    }
    read(1, cur);
    mul(0, 0, A);
#pragma unroll
    for (int i = 0; i < PPL; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, A, 0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kLgkm0);
    barrier();                                   // everybody has read this stage
    // (loads spread over the step: a wave that finds the memory pipe's queue full issues no product either)
    if (KIND == 0 || more) tall_issue_w(wo, wr, kb, cur);
    if (KIND == 2) {
      if (more) tall_issue_x<8>(p, x, kb, cur);
      mul(0, A, NM);
      mul(1, 0, NM);
      return;
    }
    mul(0, A, NM);
    mul(1, 0, B);
    if (KIND == 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, HM / 2 > 0 ? HM / 2 : 1, 0);
      }
    }
    __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (KIND == 0 || more) __builtin_amdgcn_s_waitcnt(vmcnt_imm(8));
    else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    barrier();                                   // the next stage has landed
    read(0, nxt);
    if (KIND == 0) tall_issue_x<2 * HM>(p, x, kb, cur);
    else if (more) tall_issue_x<8>(p, x, kb, cur);
    mul(1, B, NM);
    if (KIND == 0) {
#pragma unroll
      for (int i = 0; i < 2 * HM; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  using K0 = std::integral_constant<int, 0>;
  using K1 = std::integral_constant<int, 1>;
  using K2 = std::integral_constant<int, 2>;
  read(0, s0);
  for (int it = 0; it < n_it - 2; it += 2) {
    step(K0{}, it, s0, s1);
    step(K0{}, it + 1, s1, s0);
  }
  if (more) {
    tall_rows<FORM>(p, nt, x);
    wr = tall_weights<GATED>(p, nt);
  }
  step(K1{}, n_it - 2, s0, s1);
  step(K2{}, n_it - 1, s1, s0);

  // Lane: row r32 of x tile j, columns 8 q + 4 half + 0 .. 3 of W tile g in registers 4 q .. 4 q + 3.  A wave turns 32 rows at a
  // time in its 8 KB of LDS and stores whole row segments (16-byte chunk c of row r at c ^ (r & 7)).
  constexpr int CW = GATED ? 64 : 128;           // columns of a wave
  if constexpr (FORM == kTallDense) {
    if (t.slab >= 0) {
      float* const to = p.part + (int64_t)t.slab * 65536 + wn * 128 + 4 * half;
#pragma unroll
      for (int j = 0; j < HM; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4_t*>(to + (32 * (wm * HM + j) + r32) * 256 + 32 * g + 8 * q) =
                f32x4_t{acc[g][j][4 * q], acc[g][j][4 * q + 1], acc[g][j][4 * q + 2], acc[g][j][4 * q + 3]};
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
      return;
    }
  }
  char* const mine = so + wid * 8192;
  const int n0 = t.tile * (2 * CW) + wn * CW;
#pragma unroll
  for (int j = 0; j < HM; ++j) {
    const int m0 = t.row0 + 32 * (wm * HM + j);
    float pw = 1.f;
    if constexpr (FORM == MI_MOE_RELU_SQUARED) {
      if (p.pair_weights) {
        const int pr = p.row_map[m0 + r32];
        pw = pr < 0 ? 0.f : p.pair_weights[pr];
      }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
#pragma unroll
      for (int q = 0; q < (GATED ? 2 : 4); ++q) {
        float v[4], bv[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (FORM == kTallDense) {
          if (p.bias) {
            const int n = n0 + 32 * g + 8 * q + 4 * half;
            const uint2 w = *reinterpret_cast<const uint2*>(p.bias + (n < p.N ? n : 0));
            bv[0] = E::lo(w.x), bv[1] = E::hi(w.x), bv[2] = E::lo(w.y), bv[3] = E::hi(w.y);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (GATED) {      // a W tile is 16 gate rows and the up rows of the same columns
            const float gt = E::from_bits(E::to_bits(acc[g][j][4 * q + r])), up = E::from_bits(E::to_bits(acc[g][j][8 + 4 * q + r]));
            v[r] = gt / (1.f + __expf(-gt)) * up;
          } else {
            v[r] = acc[g][j][4 * q + r] + bv[r];
            if constexpr (FORM == MI_MOE_RELU_SQUARED) {
              v[r] = fmaxf(v[r] * pw, 0.f);
              v[r] *= v[r];
            }
          }
        }
        u32x2_t o = {E::pack(v[0], v[1]), E::pack(v[2], v[3])};
        const int chunk = GATED ? 2 * g + q : 4 * g + q;
        *reinterpret_cast<u32x2_t*>(mine + r32 * (2 * CW) + ((chunk ^ (r32 & 7)) << 4) + 8 * half) = o;
      }
    }
#pragma unroll
    for (int i = 0; i < CW / 16; ++i) {
      constexpr int per = CW / 8;                // 16-byte chunks of a row
      const int at = 64 * i + lane, r = at / per, c = at % per;
      const u32x4_t o = *reinterpret_cast<const u32x4_t*>(mine + r * (2 * CW) + ((c ^ (r & 7)) << 4));
      const int n = n0 + 8 * c;
      if (n < p.N && (!tall_dense(FORM) || m0 + r < p.M)) *reinterpret_cast<u32x4_t*>(p.out + (int64_t)(m0 + r) * p.ldo + n) = o;
    }
  }
  // the next item's two stages came before the stores (which a wave past the last column or row does not issue)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  if (n0 + CW <= p.N && (!tall_dense(FORM) || t.row0 + 64 * HM <= p.M)) __builtin_amdgcn_s_waitcnt(vmcnt_imm(CW / 16 * HM));
  else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
}

template <typename Tag, int FORM, bool TURN = false>
__global__ __launch_bounds__(256, 1) void tall_gemm_kernel(const TallParams p) {
  scalar_cache_acquire();
  constexpr bool GATED = tall_gated(FORM);
  __shared__ __attribute__((aligned(1024))) char s0[kTallStage];
  __shared__ __attribute__((aligned(1024))) char s1[kTallStage];
  __shared__ __attribute__((aligned(1024))) char so[32768];
  // every XCD has a contiguous range of the items, its workgroups take them in turn
  int lo, whole, tail;
  const int items = tall_items(p, tall_dense(FORM), blockIdx.x & 7, lo, whole, tail), stride = gridDim.x >> 3;
  int item = blockIdx.x >> 3;
  if (item >= items) return;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t x[8], wo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 8 * (wid + 4 * i) + (lane >> 3);
    const int n = GATED ? ((row >> 4) & 1) * p.N + 16 * (row >> 5) + (row & 15) : row;
    wo[i] = (uint32_t)n * (uint32_t)(2 * p.K) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
  TallItem t, nt;
  tall_fetch<FORM, TURN>(p, item, lo, whole, tail, t);
  tall_rows<FORM>(p, t, x);
  {
    const __amdgpu_buffer_rsrc_t wr = tall_weights<GATED>(p, t);
    tall_issue_w(wo, wr, tall_block<TURN>(t, 0), s0);
    tall_issue_x<8>(p, x, tall_block<TURN>(t, 0), s0);
    tall_issue_w(wo, wr, tall_block<TURN>(t, 1), s1);
    tall_issue_x<8>(p, x, tall_block<TURN>(t, 1), s1);
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  while (true) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    item += stride;
    const bool more = item < items;
    nt = t;
    if (more) tall_fetch<FORM, TURN>(p, item, lo, whole, tail, nt);
    if (t.units >= 4) tall_tile<Tag, FORM, TURN, 4>(p, s0, s1, so, t, x, wo, nt, more);
    else if (t.units == 3) tall_tile<Tag, FORM, TURN, 3>(p, s0, s1, so, t, x, wo, nt, more);
    else if (t.units == 2) tall_tile<Tag, FORM, TURN, 2>(p, s0, s1, so, t, x, wo, nt, more);
    else tall_tile<Tag, FORM, TURN, 1>(p, s0, s1, so, t, x, wo, nt, more);
    if (!more) break;
    t = nt;
  }
}

// the pieces' sums of a tile cut along K, in order (+ bias); a workgroup has 8 rows of a tile, a thread 8 columns
template <typename Tag>
__global__ __launch_bounds__(256) void tall_reduce_kernel(const TallParams p) {
  scalar_cache_acquire();
  using E = Elem<Tag>;
  const int cut = blockIdx.x >> 5, at = p.whole + cut;
  const int tiles = (p.M + 255) >> 8, g = at / (p.group * p.nx), in = at - g * p.group * p.nx, rows = min(p.group, tiles - p.group * g);
  const int tile = in / rows, r = 8 * (blockIdx.x & 31) + (threadIdx.x >> 5), c = 8 * (threadIdx.x & 31);
  const int m = (p.group * g + in - tile * rows) * 256 + r, n = tile * kTallN + c;
  if (m >= p.M || n >= p.N) return;
  f32x4_t v0 = {0, 0, 0, 0}, v1 = {0, 0, 0, 0};
  const float* from = p.part + (int64_t)cut * p.split * 65536 + r * 256 + c;
  for (int s = 0; s < p.split; ++s, from += 65536) {
    v0 += *reinterpret_cast<const f32x4_t*>(from);
    v1 += *reinterpret_cast<const f32x4_t*>(from + 4);
  }
  if (p.bias) {
    const uint4 b = *reinterpret_cast<const uint4*>(p.bias + n);
    v0 += f32x4_t{E::lo(b.x), E::hi(b.x), E::lo(b.y), E::hi(b.y)};
    v1 += f32x4_t{E::lo(b.z), E::hi(b.z), E::lo(b.w), E::hi(b.w)};
  }
  *reinterpret_cast<uint4*>(p.out + (int64_t)m * p.ldo + n) =
      make_uint4(E::pack(v0[0], v0[1]), E::pack(v0[2], v0[3]), E::pack(v1[0], v1[1]), E::pack(v1[2], v1[3]));
}

template <typename Tag, bool TURN>
int launch_tall_form(const TallParams& p, int form, const dim3 grid, hipStream_t s) {
  if (form == MI_MOE_GATED) hipLaunchKernelGGL((tall_gemm_kernel<Tag, MI_MOE_GATED, TURN>), grid, dim3(256), 0, s, p);
  else if (form == MI_MOE_PLAIN) hipLaunchKernelGGL((tall_gemm_kernel<Tag, MI_MOE_PLAIN, TURN>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((tall_gemm_kernel<Tag, MI_MOE_RELU_SQUARED, TURN>), grid, dim3(256), 0, s, p);
  return launch_status();
}
template <typename Tag>
int launch_tall(const TallParams& p, int form, const dim3 grid, hipStream_t s) {
  return p.turn ? launch_tall_form<Tag, true>(p, form, grid, s) : launch_tall_form<Tag, false>(p, form, grid, s);
}

}  // namespace

int launch_grouped_tall(const GroupedGemmArgs& a, hipStream_t s) {
  const bool gated = a.form == MI_MOE_GATED;
  if (a.rows_per_tile != 128 && a.rows_per_tile != 256) return MI_ERR_UNSUPPORTED;
  if (a.k % 128 || a.n_out % 16 || a.out_row_stride % 8 || ((uintptr_t)a.out & 15) || (a.dtype != MI_DTYPE_BF16 && a.dtype != MI_DTYPE_F16)) return MI_ERR_UNSUPPORTED;
  // 32-bit byte offsets into the rows (a gathered row's number is at most its pair's) and into one expert's weights
  const int64_t rows = (int64_t)a.max_tiles * a.rows_per_tile, lim = (int64_t)1 << 32;
  if (rows >= 1 << 28 || rows * a.a_row_stride * 2 >= lim || (int64_t)(gated ? 2 : 1) * a.n_out * a.k * 2 >= lim) return MI_ERR_UNSUPPORTED;
  TallParams p{};
  p.x = reinterpret_cast<const uint16_t*>(a.a_rows);
  p.w = reinterpret_cast<const uint16_t*>(a.weights);
  p.out = reinterpret_cast<uint16_t*>(a.out);
  p.N = a.n_out;
  p.K = a.k;
  p.rpt = a.rows_per_tile;
  p.gather_div = a.form != MI_MOE_PLAIN ? a.top_k : 0;
  p.div_magic = p.gather_div > 1 ? (uint32_t)((((uint64_t)1 << 32) + p.gather_div - 1) / p.gather_div) : 0;
  p.row_map = a.sorted_pairs;
  p.tile_expert = a.tile_expert;
  p.num_tiles = a.num_tiles;
  p.pair_weights = a.pair_weights;
  p.ldx = a.a_row_stride;
  p.ldo = a.out_row_stride;
  p.w_expert_stride = a.weight_expert_stride;
  p.turn = grouped_turn(a.k);
  const int cols = gated ? kTallN / 2 : kTallN;
  p.nx = (a.n_out + cols - 1) / cols;
  const int64_t work = (int64_t)p.nx * a.max_tiles;
  const dim3 grid(work < 256 ? (int)((work + 7) / 8 * 8) : 256);
  return a.dtype == MI_DTYPE_BF16 ? launch_tall<bf16_tag>(p, a.form, grid, s) : launch_tall<f16_tag>(p, a.form, grid, s);
}
}  // namespace mi

namespace {
// Tiles of one round more than fill the 256 CUs but not a whole number of rounds: the last round's tiles are cut along K so that it
// takes a fraction of a round, at the price of fp32 sums written and read.
struct TallCut {
  int tiles, whole, split;
};
TallCut tall_cut(int32_t m, int32_t n, int32_t k, bool gated) {
  TallCut c;
  const int cols = gated ? mi::kTallN / 2 : mi::kTallN;
  c.tiles = ((m + 255) / 256) * ((n + cols - 1) / cols);
  const int last = c.tiles % 256;
  c.split = last && !gated ? 256 / last : 1;
  if (c.split > k / 512) c.split = k / 512;      // at least eight blocks a piece
  if (c.split > 8) c.split = 8;
  if (c.split < 2) c.split = 1;
  c.whole = c.split > 1 ? c.tiles - last : c.tiles;
  return c;
}
bool tall_linear_ok(int32_t m, int32_t n, int32_t k, int64_t ldx, bool gated, int dtype) {
  const int64_t lim = (int64_t)1 << 32;
  return k % 128 == 0 && n % 16 == 0 && (dtype == MI_DTYPE_BF16 || dtype == MI_DTYPE_F16) && (int64_t)m * ldx * 2 < lim &&
         (int64_t)(gated ? 2 : 1) * n * k * 2 < lim;
}
}  // namespace

extern "C" int64_t mi_linear_tall_workspace_bytes(int32_t m, int32_t n, int32_t k, int32_t gated) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  const TallCut c = tall_cut(m, n, k, gated != 0);
  return c.split > 1 ? (int64_t)(c.tiles - c.whole) * c.split * 65536 * 4 : 0;
}

extern "C" int mi_linear_tall(void* out, const void* x, const void* weight, const void* bias, int32_t m, int32_t n, int32_t k,
                              int64_t x_row_stride, int64_t out_row_stride, int32_t gated, void* workspace, int64_t workspace_bytes,
                              int dtype, void* stream) {
  using namespace mi;
  if (m == 0) return MI_OK;
  if (!out || !x || !weight || m < 0 || n <= 0 || k <= 0 || (gated && bias)) return MI_ERR_INVALID_ARG;
  if (x_row_stride < k || out_row_stride < n || x_row_stride % 8 || out_row_stride % 8) return MI_ERR_INVALID_ARG;
  if (((uintptr_t)out | (uintptr_t)x | (uintptr_t)weight | (uintptr_t)bias | (uintptr_t)workspace) & 15) return MI_ERR_INVALID_ARG;
  if (!tall_linear_ok(m, n, k, x_row_stride, gated != 0, dtype)) return MI_ERR_UNSUPPORTED;
  const TallCut c = tall_cut(m, n, k, gated != 0);
  if (workspace_bytes < mi_linear_tall_workspace_bytes(m, n, k, gated) || (c.split > 1 && !workspace)) return MI_ERR_INVALID_ARG;
  TallParams p{};
  p.x = reinterpret_cast<const uint16_t*>(x);
  p.w = reinterpret_cast<const uint16_t*>(weight);
  p.out = reinterpret_cast<uint16_t*>(out);
  p.bias = reinterpret_cast<const uint16_t*>(bias);
  p.part = reinterpret_cast<float*>(workspace);
  p.M = m;
  p.N = n;
  p.K = k;
  p.rpt = 256;
  p.nx = (n + (gated ? kTallN / 2 : kTallN) - 1) / (gated ? kTallN / 2 : kTallN);
  p.whole = c.whole;
  p.split = c.split;
  p.group = 8;
  p.ldx = x_row_stride;
  p.ldo = out_row_stride;
  const int64_t items = c.whole + (int64_t)(c.tiles - c.whole) * c.split;
  const dim3 grid(items < 256 ? (int)((items + 7) / 8 * 8) : 256), block(256);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define MI_TALL(TAG)                                                                                     \
  do {                                                                                                   \
    if (gated) hipLaunchKernelGGL((tall_gemm_kernel<TAG, kTallDenseGated>), grid, block, 0, s, p);       \
    else hipLaunchKernelGGL((tall_gemm_kernel<TAG, kTallDense>), grid, block, 0, s, p);                  \
    if (c.split > 1) hipLaunchKernelGGL((tall_reduce_kernel<TAG>), dim3(32 * (c.tiles - c.whole)), block, 0, s, p); \
  } while (0)
  if (dtype == MI_DTYPE_BF16) MI_TALL(bf16_tag);
  else MI_TALL(f16_tag);
#undef MI_TALL
  return launch_status();
}
