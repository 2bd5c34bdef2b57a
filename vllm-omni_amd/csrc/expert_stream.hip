// Experts' products of a decode batch: row tiles of at most 64 rows, so that what is done is to read every chosen expert's weights
// once.  y = x W^T as D = W . x^T on the LDS images, fragments and order of sums of tall_gemm.hip (the same bits).
//
// What bounds it: HBM.  A CU has to keep about 100 KB on their way for the whole chip to read at its rate, and reads of x (from L2)
// and the turn from one tile to the next must not get in between.
//   * A workgroup per CU stays, and its tiles are one stream of 64-wide k blocks: weights are loaded three blocks ahead and x two, across
//     the border between two tiles.  Four stages of 256 weight rows and three of 64 x rows: 152 KB.
//   * Four waves, each loads a quarter of a stage and multiplies 64 weight rows by the rows of x; one barrier a block.  Fragments are
//     read with waits of their own, which leave the loads in flight alone, and the row map and the pair weights of a tile come through
//     the same stream (into 5 KB of LDS): nothing in the loop waits for memory but the count of loads in front of the barrier.
//   * Weights are read once and go past the caches (nt).  Without that a step's other launches wait for what they drove out: Pupopel decode of 253
//     at width 2048 2226 us a step, 2128 with it (the library's products 5 to 10 % each; this kernel's down product 51 -> 43).
//   * Rows without a pair, weight rows past the last one and stages past the last tile are loads past the end of a buffer: they count,
//     but read nothing.  Rows without a pair are not stored.
//   * Stores at a tile's end count like loads: the next tile's first two waits allow for them.
//   * Weight rows a multiple of 4096 bytes apart: every tile's k blocks begin with another one (StreamParams::turn), or all workgroups, which keep step
//     with each other, read from the same few channels at a time.  4096 x 1536, 200 tokens, 8 of 64, up 149 | 126 us; 2048 x 768 44.5 | 35.7.
//   * Tiles that would leave half of an XCD's workgroups idle or more in its last round are cut into halves or quarters of their weight
//     rows (expert_stream_items.h: an item of them that begins past the last column reads, multiplies and stores nothing).
// Cold weights, us, the ring kernel before | this: 64 experts of 4096 x 1536, 8 of them a token, 200 tokens, up with relu squared 172 | 126, down
// 177 | 142 (6.4 and 5.7 TB/s); 6 a token, 32 tokens, down 154 | 123; 128 experts of 1024 x 384, 512 tokens, down 27 | 23.
#include "expert_stream_items.h"
#include "mfma_attn_common.h"
#include "skinny_grouped.h"
#include "skinny_tile.h"

namespace mi {
namespace {

struct StreamParams {
  const uint16_t* x;
  const uint16_t* w;
  uint16_t* out;
  int32_t N, K;
  int32_t rpt, gather_div;      // rows per tile; > 0: source row = pair index / gather_div, else the row itself
  int32_t nx;                   // weight tiles of a row tile
  int32_t turn;                 // a tile's k blocks begin with grouped_first_block and go round
  uint32_t div_magic;           // 2^32 / gather_div, rounded up: exact for pair indices below 2^28
  uint32_t map_bytes;
  const int32_t* row_map;       // [max_rows] pair index or -1; the pairs of a tile in front
  const int32_t* tile_expert;
  const int32_t* num_tiles;     // [1]
  const float* pair_weights;    // RELU_SQUARED: the sums of a pair's row times this, in front of the activation
  int64_t ldx, ldo, w_expert_stride;
};

using lds_char = __attribute__((address_space(3))) char;

constexpr int kWStage = 32768, kXStage = 8192, kWStages = 4, kXStages = 3;
constexpr int kXRing = kWStages * kWStage, kMeta = kXRing + kXStages * kXStage;
constexpr int kMetaWave = 5 * 256;      // a wave's three row maps and two rows of pair weights
constexpr int kStreamLds = kMeta + 4 * kMetaWave;
constexpr uint32_t kDead = 0xFFFFF800u, kAll = 0xFFFFF000u;      // an offset past every buffer, a buffer's largest size

struct StreamItem {
  int row0, expert, col, cut;      // col: first output column; cut: 1, 2 or 4 items of a weight tile
};

constexpr int stream_vmcnt(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

__device__ __forceinline__ uint32_t lds_read_u32(uint32_t at) {
  uint32_t v;
  asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(at) : "memory");
  return v;
}
// fragments of two 16-wide k slices: weight rows (two tiles, 4 KB apart) and x rows
__device__ __forceinline__ void lds_read_frags(uint32_t w0, uint32_t w1, uint32_t x0, uint32_t x1, u32x4_t (&a)[2][2], u32x4_t (&b)[2][2]) {
  asm volatile(
      "ds_read_b128 %0, %8\n\t"
      "ds_read_b128 %1, %8 offset:4096\n\t"
      "ds_read_b128 %2, %9\n\t"
      "ds_read_b128 %3, %9 offset:4096\n\t"
      "ds_read_b128 %4, %10\n\t"
      "ds_read_b128 %5, %10 offset:4096\n\t"
      "ds_read_b128 %6, %11\n\t"
      "ds_read_b128 %7, %11 offset:4096\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1])
      : "v"(w0), "v"(w1), "v"(x0), "v"(x1)
      : "memory");
}

template <typename Tag, int FORM>
__global__ __launch_bounds__(256, 1) void expert_stream_kernel(const StreamParams p) {
  scalar_cache_acquire();
  using E = Elem<Tag>;
  constexpr bool GATED = FORM == MI_MOE_GATED;
  extern __shared__ __attribute__((aligned(1024))) char lds_all[];
  lds_char* const lds = (lds_char*)lds_all;      // at address 0
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // an XCD has a contiguous range of the tiles, its workgroups take them in turn
  const int per = gridDim.x >> 3, work = p.num_tiles[0] * p.nx, each = (work + 7) >> 3, lo = (blockIdx.x & 7) * each;
  const StreamSplit split = stream_split(max(min(each, work - lo), 0), per);
  const int items = split.items;
  int item = blockIdx.x >> 3;
  if (item >= items) return;
  const int n_it = p.K >> 6;

  const auto decode = [&](int i) -> StreamItem {
    StreamItem t;
    const StreamPlace q = stream_place(split, i);
    const int at = lo + q.tile, row_tile = at / p.nx;      // the weight tiles of a row tile in a row: its rows through one L2
    t.cut = q.cut;
    t.row0 = row_tile * p.rpt;
    t.expert = __builtin_amdgcn_readfirstlane(*(const __attribute__((address_space(4))) int32_t*)(p.tile_expert + row_tile));
    t.col = stream_col(q, at - row_tile * p.nx, GATED);
    return t;
  };
  const uint32_t meta = kMeta + wid * kMetaWave;
  const __amdgpu_buffer_rsrc_t map_r = __builtin_amdgcn_make_buffer_rsrc((void*)p.row_map, 0, (int)p.map_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t pw_r = __builtin_amdgcn_make_buffer_rsrc((void*)p.pair_weights, 0, (int)kAll, 0x00020000);
  const __amdgpu_buffer_rsrc_t x_r = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, (int)kAll, 0x00020000);
  const __amdgpu_buffer_rsrc_t out_r = __builtin_amdgcn_make_buffer_rsrc((void*)p.out, 0, (int)kAll, 0x00020000);
  const auto load_map = [&](int i, int slot) {
    const int row0 = (lo + stream_place(split, i).tile) / p.nx * p.rpt;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(map_r, (lds_void*)(lds + meta + 256 * slot), 4, 4 * (row0 + lane), 0, 0, 0);
  };

  uint32_t wo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 8 * (wid + 4 * i) + (lane >> 3);
    wo[i] = (uint32_t)stream_weight_row(row, p.N, GATED) * (uint32_t)(2 * p.K) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
  // ---- the loads' side of the stream: the tile that weights are loaded of, and x's offsets of it
  StreamItem lt;
  __amdgpu_buffer_rsrc_t wr = x_r;
  uint32_t xo[2], xn[2];
  int w_first = 0, x_first = 0, xn_first = 0;      // where the tiles begin along K (bytes)
  int pieces = 0, n_loaded = 0;      // n_loaded: tiles taken up so far
  const auto take = [&]() {
    const int i = item + n_loaded * per;
    if (i >= items) {
      pieces = 0;
      xn[0] = xn[1] = kDead;
      return;
    }
    lt = decode(i);
    const uint32_t map = meta + 256 * (n_loaded % 3);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 8 * (wid + 4 * h) + (lane >> 3);
      uint32_t m = lds_read_u32(map + 4 * row);
      const bool live = (int32_t)m >= 0 && row < p.rpt;
      if (p.gather_div > 1) m = __umulhi(m, p.div_magic);
      if (p.gather_div == 0) m = lt.row0 + row;
      xn[h] = live ? m * (uint32_t)(2 * p.ldx) + 16 * ((lane & 7) ^ ((row >> 1) & 7)) : kDead;
    }
    if constexpr (FORM == MI_MOE_RELU_SQUARED) {
      if (p.pair_weights) {
        const uint32_t m = lds_read_u32(map + 4 * lane);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(pw_r, (lds_void*)(lds + meta + 256 * (3 + (n_loaded & 1))), 4,
                                                 (int32_t)m >= 0 && lane < p.rpt ? 4 * m : kDead, 0, 0, 0);
      }
    }
    // weight rows past the last one read as zero and are never stored
    const StreamRange r = stream_range(lt.col, lt.cut, p.N, p.K, GATED);
    wr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w + (int64_t)lt.expert * p.w_expert_stride + r.first), 0, (int)r.bytes, 0x00020000);
    pieces = r.pieces;
    if (p.turn) w_first = xn_first = 128 * grouped_first_block(GATED, lt.expert, lt.col, p.N, n_it);
    ++n_loaded;
    if (item + n_loaded * per < items) load_map(item + n_loaded * per, n_loaded % 3);
  };
  int w_slot = 0, x_slot = 0;
  // the next blocks (bytes along K), counted from where their tile begins: with a sum of both in every block the plain form spilled twice as many
  // scalars (1024 x 384, 1 token, down 6.41 | 6.47 us)
  int w_at = 0, x_at = 0;
  const auto issue_w = [&]() {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(lds + w_slot * kWStage + (wid + 4 * i) * 1024), 16, i < pieces ? wo[i] : kDead,
                                               w_at, 0, MI_SKINNY_W_AUX);
    w_slot = (w_slot + 1) & 3;
    w_at = w_at + 128 == 128 * n_it ? 0 : w_at + 128;
    if (w_at == w_first) {
      take();
      w_at = w_first;
    }
  };
  const auto issue_x = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_r, (lds_void*)(lds + kXRing + x_slot * kXStage + (wid + 4 * i) * 1024), 16, xo[i], x_at, 0, 0);
    x_slot = x_slot == 2 ? 0 : x_slot + 1;
    x_at = x_at + 128 == 128 * n_it ? 0 : x_at + 128;
    if (x_at == x_first) {
      xo[0] = xn[0];
      xo[1] = xn[1];
      x_at = x_first = xn_first;
    }
  };

  load_map(item, 0);
  __builtin_amdgcn_s_waitcnt(stream_vmcnt(0));
  take();
  xo[0] = xn[0];
  xo[1] = xn[1];
  x_at = x_first = xn_first;
  w_at = w_first;
  StreamItem t = lt;
  issue_w();
  issue_x();
  issue_w();
  issue_x();
  issue_w();

  // ---- the products' side
  const int r32 = lane & 31, half = lane >> 5;
  uint32_t frag[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) frag[k] = r32 * 128 + ((((k & 1 ? 2 + 2 * half : 6 * half) + (k >> 1)) ^ ((r32 >> 1) & 7)) << 4);
  f32x16_t acc[2][2];
  uint32_t ws = wid * 8192, xs = kXRing;      // the stages that are read
  const int n_mine = (items - item + per - 1) / per;
  int stored = 0;      // store instructions behind the loads that the next tile's first two blocks wait for
  for (int n = 0; n < n_mine; ++n) {
    const uint32_t map = meta + 256 * (n % 3);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[g][j][i] = 0.f;
    bool work_here = wid < 4 / t.cut && t.col < p.N, upper = false;      // upper: rows 32 .. 63 hold pairs
    for (int it = 0; it < n_it; ++it) {
      // what this block needs is there when at most the two weight stages and the x stage behind it are on their way
      if (it < 2 && stored == 8) __builtin_amdgcn_s_waitcnt(stream_vmcnt(26));
      else if (it < 2 && stored == 4) __builtin_amdgcn_s_waitcnt(stream_vmcnt(22));
      else if (it < 2 && stored == 2) __builtin_amdgcn_s_waitcnt(stream_vmcnt(20));
      else __builtin_amdgcn_s_waitcnt(stream_vmcnt(18));
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (it == 0) upper = p.rpt > 32 && __builtin_amdgcn_readfirstlane((int32_t)lds_read_u32(map + 128)) >= 0;
      issue_x();
      issue_w();
      if (work_here) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          u32x4_t a[2][2], b[2][2];      // [k slice][row tile]
          lds_read_frags(ws + frag[2 * u], ws + frag[2 * u + 1], xs + frag[2 * u], xs + frag[2 * u + 1], a, b);
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int g = 0; g < 2; ++g)
              acc[g][0] = mfma32<Tag>(__builtin_bit_cast(uint4, a[k][g]), __builtin_bit_cast(uint4, b[k][0]), acc[g][0]);
          if (upper) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
              for (int g = 0; g < 2; ++g)
                acc[g][1] = mfma32<Tag>(__builtin_bit_cast(uint4, a[k][g]), __builtin_bit_cast(uint4, b[k][1]), acc[g][1]);
          }
        }
      }
      ws = ws >= 3 * kWStage ? ws - 3 * kWStage : ws + kWStage;
      xs = xs == kXRing + 2 * kXStage ? kXRing : xs + kXStage;
    }
    // Lane: row r32 of x tile j, columns 8 q + 4 half + 0 .. 3 of W tile g in registers 4 q .. 4 q + 3; the halves trade a pair of
    // q's so that each stores 16 bytes of a row
    stored = !work_here ? 0 : (upper ? 2 : 1) * (GATED ? 2 : 4);
    if (work_here) {
      const int n0 = t.col + wid * (GATED ? 32 : 64);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (j == 1 && !upper) break;
        const int row = 32 * j + r32;
        const bool live = (int32_t)lds_read_u32(map + 4 * row) >= 0 && row < p.rpt;
        float pw = 1.f;
        if constexpr (FORM == MI_MOE_RELU_SQUARED) {
          if (p.pair_weights) pw = __builtin_bit_cast(float, lds_read_u32(meta + 256 * (3 + (n & 1)) + 4 * row));
        }
        const uint32_t to = (uint32_t)(t.row0 + row) * (uint32_t)(2 * p.ldo);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
#pragma unroll
          for (int h = 0; h < (GATED ? 1 : 2); ++h) {
            uint32_t o[2][2];
#pragma unroll
            for (int qq = 0; qq < 2; ++qq) {
              const int q = 2 * h + qq;
              float v[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                if constexpr (GATED) {      // a W tile is 16 gate rows and the up rows of the same columns
                  const float gt = E::from_bits(E::to_bits(acc[g][j][4 * q + r])), up = E::from_bits(E::to_bits(acc[g][j][8 + 4 * q + r]));
                  v[r] = gt / (1.f + __expf(-gt)) * up;
                } else {
                  v[r] = acc[g][j][4 * q + r];
                  if constexpr (FORM == MI_MOE_RELU_SQUARED) {
                    v[r] = fmaxf(v[r] * pw, 0.f);
                    v[r] *= v[r];
                  }
                }
              }
              o[qq][0] = E::pack(v[0], v[1]);
              o[qq][1] = E::pack(v[2], v[3]);
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              float s0 = __builtin_bit_cast(float, o[0][c]), s1 = __builtin_bit_cast(float, o[1][c]);
              permlane32_swap(s0, s1);
              o[0][c] = __builtin_bit_cast(uint32_t, s0);
              o[1][c] = __builtin_bit_cast(uint32_t, s1);
            }
            const int col = n0 + (GATED ? 16 * g : 32 * g + 16 * h) + 8 * half;
            __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{o[0][0], o[0][1], o[1][0], o[1][1]}, out_r, live && col < p.N ? to + 2 * col : kDead, 0, 0);
          }
        }
      }
    }
    t = lt;      // the loads went on to the next tile three blocks ago
  }
  __builtin_amdgcn_s_waitcnt(stream_vmcnt(0));      // no load may land in this LDS once it is another workgroup's
}

template <typename Tag, int FORM>
int launch_stream_form(const StreamParams& p, const dim3 grid, hipStream_t s) {
  auto kern = expert_stream_kernel<Tag, FORM>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kStreamLds);
  if (attr != hipSuccess) return MI_ERR_LAUNCH;
  hipLaunchKernelGGL(kern, grid, dim3(256), kStreamLds, s, p);
  return launch_status();
}
template <typename Tag>
int launch_stream(const StreamParams& p, int form, const dim3 grid, hipStream_t s) {
  if (form == MI_MOE_GATED) return launch_stream_form<Tag, MI_MOE_GATED>(p, grid, s);
  if (form == MI_MOE_PLAIN) return launch_stream_form<Tag, MI_MOE_PLAIN>(p, grid, s);
  return launch_stream_form<Tag, MI_MOE_RELU_SQUARED>(p, grid, s);
}

}  // namespace

int launch_grouped_stream(const GroupedGemmArgs& a, hipStream_t s) {
  const bool gated = a.form == MI_MOE_GATED;
  if (a.rows_per_tile != 32 && a.rows_per_tile != 64) return MI_ERR_UNSUPPORTED;
  // the loads run three blocks ahead: at most into the next tile
  if (a.k % 64 || a.k < 256 || a.n_out % 16 || a.out_row_stride % 8 || ((uintptr_t)a.out & 15) || (a.dtype != MI_DTYPE_BF16 && a.dtype != MI_DTYPE_F16))
    return MI_ERR_UNSUPPORTED;
  // 32-bit byte offsets into the rows (a gathered row's number is at most its pair's), one expert's weights, the pairs' weights and the output
  const int64_t rows = (int64_t)a.max_tiles * a.rows_per_tile, lim = (int64_t)kAll;
  if (rows >= 1 << 28 || rows * a.a_row_stride * 2 >= lim || rows * a.out_row_stride * 2 >= lim || (int64_t)(gated ? 2 : 1) * a.n_out * a.k * 2 >= lim)
    return MI_ERR_UNSUPPORTED;
  StreamParams p{};
  p.x = reinterpret_cast<const uint16_t*>(a.a_rows);
  p.w = reinterpret_cast<const uint16_t*>(a.weights);
  p.out = reinterpret_cast<uint16_t*>(a.out);
  p.N = a.n_out;
  p.K = a.k;
  p.rpt = a.rows_per_tile;
  p.gather_div = a.form != MI_MOE_PLAIN ? a.top_k : 0;
  p.div_magic = p.gather_div > 1 ? (uint32_t)((((uint64_t)1 << 32) + p.gather_div - 1) / p.gather_div) : 0;
  p.map_bytes = (uint32_t)(rows * 4);
  p.row_map = a.sorted_pairs;
  p.tile_expert = a.tile_expert;
  p.num_tiles = a.num_tiles;
  p.pair_weights = a.pair_weights;
  p.ldx = a.a_row_stride;
  p.ldo = a.out_row_stride;
  p.w_expert_stride = a.weight_expert_stride;
  const int cols = gated ? kStreamRows / 2 : kStreamRows;
  p.nx = (a.n_out + cols - 1) / cols;
  p.turn = grouped_turn(a.k);
  const dim3 grid(256);
  return a.dtype == MI_DTYPE_BF16 ? launch_stream<bf16_tag>(p, a.form, grid, s) : launch_stream<f16_tag>(p, a.form, grid, s);
}
}  // namespace mi
