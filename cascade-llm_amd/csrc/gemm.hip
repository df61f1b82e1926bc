// MFMA bf16 GEMM family for prefill (M = prompt tokens > 1) on gfx950.
//
//   Y[M, N] = epilogue(X[M, K] . W[N, K]^T)
//
// X holds the (already RMS-normalised) token rows, W is a weight matrix in
// the reference's row-major [out_features, in_features] layout, so both
// operands are read along K.  This replaces F.linear with a [1, S, 4096]
// input (layer_streaming/llama31.py:241-279 during the prefill call, and the
// resident LM head, llama31.py:330-334).
//
// Tiling.  A workgroup computes a BM x 128 output tile (or two side by
// side), K walked in 64-deep slabs; each
// wave owns 64 (or 128) rows x 64 (or 32) columns of
// v_mfma_f32_16x16x32_bf16 fragments and reads its A and B fragments (16
// bytes a lane) from LDS.  Shapes (launch_gemm picks one):
//   GemmTileWide 256 x 256 (two 128-column sub-tiles), 8 waves of 128 x 64,
//                64-deep slabs in two buffers (gemm_wide_run): where its
//                schedule of rounds is shorter than GemmTile256's;
//   GemmTile160  160 x 256 (two sub-tiles), 8 waves of 80 x 64, a ring of 3:
//                prompts that fill 160-row tiles better than 256-row ones
//                (129 .. 160, 257 .. 320, 513 .. 640 rows), and split K
//                where its tiles divide over the CUs more evenly;
//   GemmTile256  256 x 128, 8 waves, a ring of 3 slab buffers: the other
//                GEMMs of at least as many 256-row tiles as CUs (q, o, down
//                and the fused q|k|v at M = 2048);
//   GemmTile128  128 x 128, 4 waves, a ring of 4;
//   GemmTile64   64 x 128, 4 waves, a ring of 6: where 128-row tiles would
//                leave CUs idle (the N = 1024 K / V projections at M = 2048).
// Prompts of up to 160 or 256 rows run gemm_stream.hip instead.
// When the last round of tiles would leave at least half of the CUs idle,
// the last tile columns run as tiles of half the height in the same launch
// (GemmTileWideHalf, 128 x 256, for GemmTileWide; GemmTile128x8 for
// GemmTile256; GemmTile64 for GemmTile128): the fused gate|up (28672 weight
// rows) at M = 2048 runs 768 of its 896 256 x 256 tiles in three rounds, then
// 256 half tiles, instead of three and a half rounds of full tiles.
//
// Staging.  Slabs move global -> LDS by buffer loads that write LDS
// themselves (buffer_load_dwordx4 ... lds: no staging registers, no
// ds_write), issued from inline asm (dma_lds16) so that the compiler, which
// cannot tell which ring buffer such a load writes, adds no waits of its
// own.  Slab s lives in ring buffer s % STAGES.  Step s waits (explicit
// vmcnt) for this wave's loads of slab s + 1 only, one barrier publishes
// slab s + 1 and frees slab s's buffer, the first MFMAs of slab s issue,
// and the rest of the step runs in chunks, one per load instruction of
// slab s + STAGES (into the freed buffer): each chunk issues its load, then
// its share of slab s's MFMAs interleaved with its share of slab s + 1's
// fragment reads.  The MFMAs run from the registers filled one step
// earlier, so they never wait on an LDS read; and the loads leave one at a
// time over the step instead of all eight waves queueing theirs at the
// CU's load path right after the barrier, where a wave stuck behind its
// own burst held up its MFMAs (M = 2048, rotating weights, same bits:
// q/o_proj 61.3 -> 55.7 us, down_proj 190.5 -> 185.9, q|k|v-shaped
// N = 6144 95.8 -> 85.2, fused gate|up 407.0 -> 395.1).
//
// LDS layout of a slab: 128-byte rows (64 bf16) back to back; 16-byte
// chunk c of row r sits at chunk c ^ ((r / 2) % 8).  A fragment read (16
// lanes: 16 consecutive rows, one chunk) then hits 16 distinct 16-byte bank
// groups, each read is a per-lane base plus an immediate offset, and a load
// instruction (64 lanes x 16 bytes) fills 8 whole rows, so its lanes read
// whole 128-byte row segments.  Rows past m (X) or past a matrix's rows (W)
// read as zeros through the buffer bounds; their results are not stored.
//
// A wave's columns are not contiguous: its first-half fragments and its
// second-half fragments sit 64 columns apart, so fragment j and j + H of
// one lane hold columns c and c + 64.  That pairs the two halves of a head
// (RoPE's rotate_half) and, with gate rows in tile columns 0..63 and up
// rows in 64..127, a gate and its up value, so those epilogues need no data
// exchange.
//
// Tile order.  Workgroups are dispatched round-robin over the 8 XCDs (each
// with its own L2); workgroup b runs logical tile (b % 8) * (grid / 8) +
// b / 8, so an XCD walks a contiguous range of logical tiles, which are
// ordered in groups of 4 M-tiles (column-major inside a group).  A round of
// an XCD's 32 CUs then covers a 4 x 8 block of tiles, which loads each X
// slab line 8 times and each W slab line 4 times from the XCD's L2 (83% hit
// at best, against 79% for 8 x 4; measured 1-2% faster on q, down_proj,
// q|k|v and gate|up at M = 2048).
//
// Epilogues reproduce the reference's bf16 rounding points (the GEMV family
// in gemv.hip applies the same ones):
//   store     y = bf16(acc)                               F.linear
//   residual  y = bf16(res + bf16(acc))                   residual + F.linear
//   qkv_rope  q/k heads: bf16 RoPE at position pos0 + row, then the q rows
//             or the layer's KV cache at slot slot0 + row;  v heads: cache
//   swiglu    bf16(bf16(silu(bf16(g))) * bf16(u))
//   silu / mul  the matrix-granularity halves of swiglu
//   f32       fp32 output (LM-head logits, not rounded)
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "gemm_common.h"

namespace cascade {

constexpr int kTileN = 128;
constexpr int kTileK = 64;
constexpr int kGroupM = 4;

// Tile (tm, tn) of logical tile t in a tiles_m x tiles_n grid (false:
// padding workgroup, no work).  Logical tiles run in groups of kGroupM
// tile rows, column-major inside a group.
__device__ __forceinline__ bool gemm_tile(int t, int tiles, int tiles_m, int tiles_n,
                                          int &tm, int &tn) {
  if (t >= tiles) return false;
  const int group_size = kGroupM * tiles_n;
  const int group = t / group_size;
  const int first = group * kGroupM;
  const int gm = min(kGroupM, tiles_m - first);
  const int r = t - group * group_size;
  tm = first + r % gm;
  tn = r / gm;
  return true;
}

// Tile shapes.  A tile is NSUB sub-tiles of 128 columns side by side (a
// sub-tile is one head of q|k|v, or 64 gate + 64 up rows); the BM rows of a
// sub-tile are split over WM x WN waves, each owning FM x FN fragments of
// 16 x 16.
template <int BM_, int WM_, int WN_, int NSUB_ = 1>
struct GemmTile {
  static constexpr int BM = BM_;
  static constexpr int WM = WM_;
  static constexpr int WN = WN_;
  static constexpr int NSUB = NSUB_;
  static constexpr int BN = kTileN * NSUB;
  static constexpr int SUBWAVES = WM * WN;  // waves of one sub-tile
  static constexpr int WAVES = SUBWAVES * NSUB;
  static constexpr int FM = BM / WM / 16;
  static constexpr int FN = kTileN / WN / 16;
  static constexpr int H = FN / 2;  // fragments per half sub-tile
  // staged epilogue: bf16 per staged column (BM rows + 8 pad; the column
  // stride is 4 banks mod 64, so 16 lanes writing 16 columns hit 16
  // distinct 4-bank groups)
  static constexpr int STAGE_COL = BM + 8;
  static_assert(WAVES == 4 || WAVES == 8, "4 or 8 waves");
};
using GemmTile256 = GemmTile<256, 4, 2>;  // 8 waves of 64 x 64
using GemmTile128 = GemmTile<128, 2, 2>;  // 4 waves of 64 x 64
using GemmTile64 = GemmTile<64, 1, 4>;    // 4 waves of 64 x 32
using GemmTile128x8 = GemmTile<128, 2, 4>;  // 8 waves of 64 x 32 (half of GemmTile256)
using GemmTileWide = GemmTile<256, 2, 2, 2>;      // 8 waves of 128 x 64, 256 columns
using GemmTileWideHalf = GemmTile<128, 2, 2, 2>;  // 8 waves of 64 x 64, 256 columns
using GemmTile160 = GemmTile<160, 2, 2, 2>;       // 8 waves of 80 x 64, 256 columns

// Tile column of fragment j of wave column wn for lane row lr.  A wave's
// first-half fragments (j < H) and second-half fragments (j >= H) sit 64
// columns apart, so fragment j and j + H of one lane hold columns c and
// c + 64: the two halves of a RoPE head, or a gate row and its up row.
template <class T>
__device__ __forceinline__ int gemm_col(int wn, int j, int lr) {
  return 16 * T::H * wn + 16 * (j % T::H) + 64 * (j / T::H) + lr;
}

template <int EPI, class T>
__device__ __forceinline__ void gemm_epilogue(
    const GemmArgs &a, int tm, int tn, int wm, int wn, int lane,
    const f32x4 (&acc)[T::FM][T::FN]) {
  const int lr = lane & 15;
  const int lq = lane >> 4;
#pragma unroll
  for (int i = 0; i < T::FM; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t row = static_cast<int64_t>(tm) * T::BM +
                          (T::BM / T::WM) * wm + 16 * i + 4 * lq + r;
      if (row >= a.m) continue;
      if constexpr (EPI == kGemmQkvRope) {
        const int64_t hq = a.n0 / kGemmHead, hk = a.n1 / kGemmHead;
        const int64_t pos = a.pos0 + row;
#pragma unroll
        for (int j = 0; j < T::H; ++j) {
          const int d = gemm_col<T>(wn, j, lr);  // 0..63
          const float xa = round_bf16(acc[i][j][r]);
          const float xb = round_bf16(acc[i][j + T::H][r]);
          uint16_t oa, ob;
          if (tn < hq + hk) {
            // x*cos + rotate_half(x)*sin, products and sum rounded to bf16
            // (apply_rotary_pos_emb on bf16 tensors)
            const float c = bf16_to_f32(a.rope_cos[pos * kGemmHalfHead + d]);
            const float s = bf16_to_f32(a.rope_sin[pos * kGemmHalfHead + d]);
            oa = f32_to_bf16(round_bf16(xa * c) + round_bf16(-xb * s));
            ob = f32_to_bf16(round_bf16(xb * c) + round_bf16(xa * s));
          } else {
            oa = f32_to_bf16(xa);
            ob = f32_to_bf16(xb);
          }
          uint16_t *dst;
          if (tn < hq) {
            dst = a.y + row * a.ldy + static_cast<int64_t>(tn) * kGemmHead;
          } else if (tn < hq + hk) {
            dst = a.k_out + (tn - hq) * a.kv_head_stride +
                  (a.slot0 + row) * kGemmHead;
          } else {
            dst = a.v_out + (tn - hq - hk) * a.kv_head_stride +
                  (a.slot0 + row) * kGemmHead;
          }
          dst[d] = oa;
          dst[d + kGemmHalfHead] = ob;
        }
      } else if constexpr (EPI == kGemmSwiglu) {
#pragma unroll
        for (int j = 0; j < T::H; ++j) {
          const int64_t col =
              static_cast<int64_t>(tn) * kGemmHalfHead + gemm_col<T>(wn, j, lr);
          const float g = round_bf16(acc[i][j][r]);
          const float u = round_bf16(acc[i][j + T::H][r]);
          const float s = round_bf16(gemm_silu(g));
          a.y[row * a.ldy + col] = f32_to_bf16(s * u);
        }
      } else {
#pragma unroll
        for (int j = 0; j < T::FN; ++j) {
          const int64_t col =
              static_cast<int64_t>(tn) * kTileN + gemm_col<T>(wn, j, lr);
          if (col >= a.n0) continue;
          const int64_t at = row * a.ldy + col;
          if constexpr (EPI == kGemmF32) {
            a.yf[at] = acc[i][j][r];
            continue;
          }
          const float v = round_bf16(acc[i][j][r]);
          float out;
          if constexpr (EPI == kGemmStore) {
            out = v;
          } else if constexpr (EPI == kGemmResidual) {
            out = bf16_to_f32(a.aux[at]) + v;
          } else if constexpr (EPI == kGemmSilu) {
            out = gemm_silu(v);
          } else {  // kGemmMul
            out = bf16_to_f32(a.aux[at]) * v;
          }
          a.y[at] = f32_to_bf16(out);
        }
      }
    }
  }
}

// Vectorised epilogue.  The waves first write their fragments to LDS in
// column-major order (a lane's 4 rows of one column are 8 contiguous bytes:
// one ds_write_b64 per fragment), then read them back row-major with
// ds_read_b64_tr_b16, which hands lane i of a 16-lane group row i of the 4
// columns the group addresses, so every lane ends up with 8 consecutive
// columns of one row and loads aux / stores results 16 bytes at a time.
// Column stride (BM + 8) bf16 (GemmTile::STAGE_COL): the fragment writes
// of a lane group fall in distinct banks.  The values staged are those of
// the direct epilogue's rounding points (bf16(acc), or the final SwiGLU
// product), so results are the same bit for bit.

__device__ __forceinline__ uint2 stage_read_tr(const uint16_t *p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  const s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4 *)(p));
  return __builtin_bit_cast(uint2, r);
}

__device__ __forceinline__ float lo_f(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float hi_f(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }

template <int EPI, class T>
__device__ __forceinline__ void gemm_epilogue_staged(
    const GemmArgs &a, int tm, int tn, int wm, int wn, int lane, int wave,
    const f32x4 (&acc)[T::FM][T::FN], uint16_t *stage) {
  const int lr = lane & 15;
  const int lq = lane >> 4;
  const int arow = (T::BM / T::WM) * wm;
  // items: 16 rows x 32 columns of the output sub-tile; lane (g, i) of a
  // wave takes row i, columns 8 g .. 8 g + 7 of the item.  Wave w of the
  // sub-tile takes items w, w + SUBWAVES, ...
  constexpr int TW = EPI == kGemmSwiglu || EPI == kGemmQkvRope ? 64 : kTileN;
  constexpr int kItems = (T::BM / 16) * (TW / 32);
  constexpr int kPer = kItems / T::SUBWAVES;
  static_assert(kItems % T::SUBWAVES == 0, "whole items per wave");
  const int g = lq, li = lr;
  auto item_r0 = [&](int n) { return 16 * ((wave + T::SUBWAVES * n) / (TW / 32)); };
  auto item_c0 = [&](int n) { return 32 * ((wave + T::SUBWAVES * n) % (TW / 32)) + 8 * g; };
  const int64_t ncols = a.n0;  // output width (SwiGLU: n_half)

  // ---- inputs the epilogue reads from memory, issued first so their
  // latency overlaps the staging below
  u32x4 in0[kPer], in1[kPer];
#pragma unroll
  for (int n = 0; n < kPer; ++n) {
    const int64_t row = static_cast<int64_t>(tm) * T::BM + item_r0(n) + li;
    in0[n] = in1[n] = u32x4{0u, 0u, 0u, 0u};
    if (row >= a.m) continue;
    if constexpr (EPI == kGemmResidual || EPI == kGemmMul) {
      const int64_t col = static_cast<int64_t>(tn) * TW + item_c0(n);
      if (col + 8 <= ncols)
        in0[n] = *reinterpret_cast<const u32x4 *>(a.aux + row * a.ldy + col);
    } else if constexpr (EPI == kGemmQkvRope) {
      if (tn < (a.n0 + a.n1) / kGemmHead) {
        const int64_t pos = a.pos0 + row;
        in0[n] = *reinterpret_cast<const u32x4 *>(a.rope_cos + pos * kGemmHalfHead + item_c0(n));
        in1[n] = *reinterpret_cast<const u32x4 *>(a.rope_sin + pos * kGemmHalfHead + item_c0(n));
      }
    }
  }

  // ---- fragments -> LDS (column-major, 4 rows per 8-byte piece)
  if constexpr (EPI == kGemmSwiglu) {
    // column c (0..63) holds bf16(silu(bf16(gate c)) * bf16(up c))
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
      for (int j = 0; j < T::H; ++j) {
        const int col = gemm_col<T>(wn, j, lr);
        uint2 v;
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float gt = round_bf16(acc[i][j][r]);
          const float u = round_bf16(acc[i][j + T::H][r]);
          o[r] = round_bf16(gemm_silu(gt)) * u;
        }
        v.x = pack_bf16x2(o[0], o[1]);
        v.y = pack_bf16x2(o[2], o[3]);
        *reinterpret_cast<uint2 *>(stage + col * T::STAGE_COL + arow + 16 * i + 4 * lq) = v;
      }
  } else {
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
      for (int j = 0; j < T::FN; ++j) {
        const int col = gemm_col<T>(wn, j, lr);
        uint2 v;
        v.x = pack_bf16x2(acc[i][j][0], acc[i][j][1]);
        v.y = pack_bf16x2(acc[i][j][2], acc[i][j][3]);
        *reinterpret_cast<uint2 *>(stage + col * T::STAGE_COL + arow + 16 * i + 4 * lq) = v;
      }
  }
  __syncthreads();

  // ---- LDS -> rows
  const int qk = li >> 2, qq = li & 3;  // addressing lane k = 4 j + q of the group
  auto read8 = [&](int r0, int c0, uint32_t (&w)[4]) {
    // two transposed reads: columns c0 .. c0 + 3 and c0 + 4 .. c0 + 7
    const uint2 lo = stage_read_tr(stage + (c0 + qk) * T::STAGE_COL + r0 + 4 * qq);
    const uint2 hi = stage_read_tr(stage + (c0 + 4 + qk) * T::STAGE_COL + r0 + 4 * qq);
    w[0] = lo.x; w[1] = lo.y; w[2] = hi.x; w[3] = hi.y;
  };
#pragma unroll
  for (int n = 0; n < kPer; ++n) {
    const int r0 = item_r0(n), c0 = item_c0(n);
    const int64_t row = static_cast<int64_t>(tm) * T::BM + r0 + li;
    // the transposed reads need every addressing lane: read before any
    // lane drops out
    uint32_t w[4], w2[4];
    read8(r0, c0, w);  // bf16 pairs: columns c0 + 2 p, c0 + 2 p + 1
    if constexpr (EPI == kGemmQkvRope) read8(r0, c0 + kGemmHalfHead, w2);  // d + 64
    if (row >= a.m) continue;
    if constexpr (EPI == kGemmQkvRope) {
      const int64_t hq = a.n0 / kGemmHead, hk = a.n1 / kGemmHead;
      u32x4 oa, ob;
      if (tn < hq + hk) {
        const u32x4 cs = in0[n], sn = in1[n];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          // x*cos + rotate_half(x)*sin, products and sum rounded to bf16
          const float xa0 = lo_f(w[p]), xa1 = hi_f(w[p]);
          const float xb0 = lo_f(w2[p]), xb1 = hi_f(w2[p]);
          const float c0f = lo_f(cs[p]), c1f = hi_f(cs[p]);
          const float s0f = lo_f(sn[p]), s1f = hi_f(sn[p]);
          oa[p] = pack_bf16x2(round_bf16(xa0 * c0f) + round_bf16(-xb0 * s0f),
                              round_bf16(xa1 * c1f) + round_bf16(-xb1 * s1f));
          ob[p] = pack_bf16x2(round_bf16(xb0 * c0f) + round_bf16(xa0 * s0f),
                              round_bf16(xb1 * c1f) + round_bf16(xa1 * s1f));
        }
      } else {
        oa = u32x4{w[0], w[1], w[2], w[3]};
        ob = u32x4{w2[0], w2[1], w2[2], w2[3]};
      }
      uint16_t *dst;
      if (tn < hq) {
        dst = a.y + row * a.ldy + static_cast<int64_t>(tn) * kGemmHead;
      } else if (tn < hq + hk) {
        dst = a.k_out + (tn - hq) * a.kv_head_stride + (a.slot0 + row) * kGemmHead;
      } else {
        dst = a.v_out + (tn - hq - hk) * a.kv_head_stride + (a.slot0 + row) * kGemmHead;
      }
      *reinterpret_cast<u32x4 *>(dst + c0) = oa;
      *reinterpret_cast<u32x4 *>(dst + c0 + kGemmHalfHead) = ob;
    } else {
      const int64_t col = static_cast<int64_t>(tn) * TW + c0;
      const int64_t at = row * a.ldy + col;
      u32x4 out;
      if constexpr (EPI == kGemmStore || EPI == kGemmSwiglu) {
        out = u32x4{w[0], w[1], w[2], w[3]};
      } else {
        const u32x4 aux = in0[n];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const float v0 = lo_f(w[p]), v1 = hi_f(w[p]);
          float o0, o1;
          if constexpr (EPI == kGemmResidual) {
            o0 = lo_f(aux[p]) + v0; o1 = hi_f(aux[p]) + v1;
          } else if constexpr (EPI == kGemmSilu) {
            o0 = gemm_silu(v0); o1 = gemm_silu(v1);
          } else {  // kGemmMul
            o0 = lo_f(aux[p]) * v0; o1 = hi_f(aux[p]) * v1;
          }
          out[p] = pack_bf16x2(o0, o1);
        }
      }
      if (col + 8 <= ncols) {
        *reinterpret_cast<u32x4 *>(a.y + at) = out;
      } else if (col < ncols) {  // N tail: element stores (aux read element-wise)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (col + e >= ncols) break;
          const uint32_t pr = w[e >> 1];
          const float v = (e & 1) ? hi_f(pr) : lo_f(pr);
          float o = v;
          if constexpr (EPI == kGemmResidual) o = bf16_to_f32(a.aux[at + e]) + v;
          else if constexpr (EPI == kGemmSilu) o = gemm_silu(v);
          else if constexpr (EPI == kGemmMul) o = bf16_to_f32(a.aux[at + e]) * v;
          a.y[at + e] = f32_to_bf16(o);
        }
      }
    }
  }
}

// Slab geometry (see the staging and layout notes at the top).
template <int BK>
struct DmaSlab {
  static constexpr int CH = BK / 8;         // 16-byte chunks per row
  static constexpr int ROWB = 2 * BK;       // bytes per row
  static constexpr int RPB = 256 / ROWB;    // rows per 256-byte bank cycle
  static constexpr int RPI = 1024 / ROWB;   // rows per load instruction
  static_assert(BK == 32 || BK == 64, "slab depth");
};

// Ring geometry of a tile shape: bf16 elements of one slab buffer (X rows,
// then W rows), and of the LDS a workgroup needs (the ring, or the staged
// output tile of the vectorised epilogue, which reuses it).
template <class T, int STAGES, int BK = kTileK>
struct GemmRing {
  static constexpr int XB = T::BM * BK;
  static constexpr int WB = T::BN * BK;
  static constexpr int SLAB = XB + WB;
  static constexpr int STAGE = T::NSUB * kTileN * T::STAGE_COL;
  static constexpr int LDS = STAGES * SLAB > STAGE ? STAGES * SLAB : STAGE;
};

// The matrix of q|k|v head h, its rows and the head's first row in it.
struct HeadRows {
  const uint16_t *base;
  int64_t rows, row;
};
__device__ __forceinline__ HeadRows head_rows(const GemmArgs &a, int64_t h) {
  const int64_t hq = a.n0 / kGemmHead, hk = a.n1 / kGemmHead;
  if (h < hq) return {a.w0, a.n0, h * kGemmHead};
  if (h < hq + hk) return {a.w1, a.n1, (h - hq) * kGemmHead};
  return {a.w2, a.n2, (h - hq - hk) * kGemmHead};
}

// Output tile (tm, tn) of shape T: rows tm * BM .., 128-column sub-tiles
// tn * NSUB .. (q|k|v: head tn; SwiGLU: gate / up rows 64 per sub-tile).
// sb0 holds the ring.
template <int EPI, class T, int STAGES, int BK = kTileK>
__device__ __forceinline__ void gemm_tile_run(const GemmArgs &a, int tm, int tn,
                                              uint16_t *sb0) {
  static_assert(STAGES >= 3, "a ring of at least 3 slab buffers");
  using L = DmaSlab<BK>;
  using R = GemmRing<T, STAGES, BK>;
  constexpr int XI = T::BM * L::ROWB / 1024;  // load instructions per X slab
  constexpr int WI = T::BN * L::ROWB / 1024;
  // per wave; 160-row tiles leave waves XR .. 7 one X load fewer than the
  // others (the last of the XW, and of every vmcnt below)
  constexpr int XW = (XI + T::WAVES - 1) / T::WAVES, WW = WI / T::WAVES;
  constexpr int XR = XI % T::WAVES;
  static_assert(WI % T::WAVES == 0, "whole W loads per wave");
  constexpr int XB = R::XB, kSlab = R::SLAB;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const bool more = XR == 0 || wave < XR;  // issues all XW of its X loads
  const int sub = wave / T::SUBWAVES;  // sub-tile of the wave
  const int sw = wave % T::SUBWAVES;
  const int wm = sw / T::WN;
  const int wn = sw % T::WN;
  const int lr = lane & 15;
  const int g4 = lane >> 4;
  const int64_t k_bytes = a.k * 2;

  // operands as buffer resources; W instruction i reads matrix wsel(i)
  const uint16_t *wbase0, *wbase1;
  int64_t wrows0, wrows1, wrow0, wrow1;  // rows of each matrix, first tile row in it
  if constexpr (EPI == kGemmSwiglu) {
    wbase0 = a.w0; wrows0 = a.n0; wrow0 = static_cast<int64_t>(tn) * T::NSUB * kGemmHalfHead;
    wbase1 = a.w1; wrows1 = a.n0; wrow1 = wrow0;
  } else if constexpr (EPI == kGemmQkvRope) {
    // one head per sub-tile
    const HeadRows h0 = head_rows(a, static_cast<int64_t>(tn) * T::NSUB);
    const HeadRows h1 = head_rows(a, static_cast<int64_t>(tn) * T::NSUB + T::NSUB - 1);
    wbase0 = h0.base; wrows0 = h0.rows; wrow0 = h0.row;
    wbase1 = h1.base; wrows1 = h1.rows; wrow1 = h1.row;
  } else {
    wbase0 = a.w0; wrows0 = a.n0; wrow0 = static_cast<int64_t>(tn) * T::BN;
    wbase1 = wbase0; wrows1 = wrows0; wrow1 = wrow0;
  }
  const u32x4 xw = buffer_rsrc_words(a.x, a.m * k_bytes);
  const u32x4 ww0 = buffer_rsrc_words(wbase0, wrows0 * k_bytes);
  const u32x4 ww1 = buffer_rsrc_words(wbase1, wrows1 * k_bytes);

  // lane part of a load: row L / CH of the instruction's RPI rows, physical
  // chunk L % CH, i.e. logical chunk (L % CH) ^ f(row); f depends on the
  // instruction only through its parity (BK = 64)
  const int ld_r = lane / L::CH;
  auto ld_off = [&](int parity) {
    const int f = ((L::RPI * parity + ld_r) / L::RPB) % L::CH;
    return ld_r * static_cast<int>(k_bytes) + 16 * ((lane % L::CH) ^ f);
  };
  const int ld_off0 = ld_off(0), ld_off1 = ld_off(1);

  // fragment reads: rows 16 q + lr (q: fragment), chunk 4 ks + g4 at
  // physical chunk (4 ks + g4) ^ f(lr), f(lr) = (lr / RPB) % CH
  const int fl = (lr / L::RPB) % L::CH;
  const int rd_off0 = lr * L::ROWB + 16 * ((g4) ^ fl);
  const int rd_off1 = lr * L::ROWB + 16 * ((4 + g4) ^ fl);
  const int arow0 = (T::BM / T::WM) * wm;

  f32x4 acc[T::FM][T::FN];
#pragma unroll
  for (int i = 0; i < T::FM; ++i)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const int slab0 = a.split_slabs ? static_cast<int>(blockIdx.y) * a.split_slabs : 0;
  const int slabs = a.split_slabs ? min(a.split_slabs, static_cast<int>(a.k / BK) - slab0)
                                  : static_cast<int>(a.k / BK);
  // LDS byte address of sb0 (the ring's buffer b starts kSlab * 2 b bytes
  // later)
  const uint32_t ring_lds = lds_address(sb0);
  // The whole byte offset goes in voffset: the buffer range check covers
  // voffset (not soffset), so rows past the end read as zeros instead of
  // leaving the allocation.  Offsets stay below 2^31 (checked on the host).
  // Load instruction h (0 .. XW + WW - 1) of this wave for slab `slab`
  // into ring buffer `buf`: X rows first, then W rows.
  auto ring_load_one = [&](int slab, int buf, int h) __attribute__((always_inline)) {
    const uint32_t dx = ring_lds + static_cast<uint32_t>(buf * kSlab * 2);
    const uint32_t dw = dx + XB * 2;
    const int kb = (slab0 + slab) * BK * 2;
    if (h < XW) {
      if (h == XW - 1 && !more) return;
      const int i = XR ? wave + T::WAVES * h : wave * XW + h;
      const int64_t row = static_cast<int64_t>(tm) * T::BM + L::RPI * i;
      dma_lds16(xw, ((i & 1) ? ld_off1 : ld_off0) + static_cast<int>(row * k_bytes) + kb,
                dx + i * 1024);
    } else {
      const int i = wave * WW + (h - XW);
      const int trow = L::RPI * i;  // tile row of the instruction
      // SwiGLU: sub-tile trow / 128 holds 64 gate rows, then their 64 up rows
      const int tt = trow % kTileN;
      const bool second = EPI == kGemmSwiglu    ? tt >= kGemmHalfHead
                          : EPI == kGemmQkvRope ? trow >= kTileN
                                                : false;
      const int64_t row =
          EPI == kGemmSwiglu
              ? (second ? wrow1 : wrow0) + (trow / kTileN) * kGemmHalfHead + tt % kGemmHalfHead
          : EPI == kGemmQkvRope ? (second ? wrow1 : wrow0) + tt
                                : wrow0 + trow;
      dma_lds16(second ? ww1 : ww0,
                ((i & 1) ? ld_off1 : ld_off0) + static_cast<int>(row * k_bytes) + kb,
                dw + i * 1024);
    }
  };
  auto ring_load = [&](int slab, int buf) {
#pragma unroll
    for (int h = 0; h < XW + WW; ++h) ring_load_one(slab, buf, h);
  };
  // Slab j lives in ring buffer j % STAGES.  Step s (one per slab):
  //   wait for this wave's loads of slab s + 1 (the loads of the
  //   STAGES - 2 slabs after it may stay in flight) and for its LDS reads
  //   of slab s (lgkmcnt 0); one barrier publishes slab s + 1 and frees
  //   slab s's buffer;
  //   slab s + STAGES goes out into that buffer, one load instruction at
  //   the head of each of the step's D chunks;
  //   slab s + 1's fragments are read into registers while slab s's
  //   MFMAs, whose fragments were read one step earlier, run: the MFMA
  //   queue never waits on an LDS read.
  // Steps past the end reload the last slab and read fragments that are
  // never used, so every step issues the same loads and a constant vmcnt
  // covers every wait.
  constexpr int D = XW + WW;
  constexpr int kAhead = (STAGES - 2) * D;
  constexpr int kAheadFirst = (STAGES - 1) * D;
  static_assert(kAheadFirst < 64, "vmcnt holds 6 bits");
  constexpr int kWaitAll = waitcnt_imm(0, 0);
  constexpr int KS = BK / 32;
  constexpr int kReads = KS * (T::FM + T::FN);
  constexpr int kMfmas = KS * T::FM * T::FN;
  // MFMAs issued right after the step barrier (at most 4, leaving one MFMA
  // for every fragment read in the chunks after them)
  constexpr int kLead = kMfmas - kReads < 4 ? kMfmas - kReads : 4;
  constexpr int kRest = kMfmas - kLead;
  // every chunk holds at least as many MFMAs as fragment reads
  static_assert(kRest >= kReads && kRest / D >= (kReads + D - 1) / D,
                "one MFMA ahead of every fragment read in each chunk");
  using FragA = u32x4[KS][T::FM];
  using FragB = u32x4[KS][T::FN];
  // Fragment read r (0 .. kReads - 1) of slab buffer `buf`: for each
  // 32-deep half ks of the slab, the FM A fragments, then the FN B ones.
  auto read_frag = [&](int buf, int r, FragA &fa, FragB &fb) __attribute__((always_inline)) {
    const char *ax = reinterpret_cast<const char *>(sb0 + buf * kSlab) + arow0 * L::ROWB;
    const char *aw = reinterpret_cast<const char *>(sb0 + buf * kSlab + XB);
    const int ks = r / (T::FM + T::FN), q = r % (T::FM + T::FN);
    const int off = ks ? rd_off1 : rd_off0;
    if (q < T::FM) {
      fa[ks][q] = *reinterpret_cast<const u32x4 *>(ax + off + 16 * q * L::ROWB);
    } else {
      const int j = q - T::FM;
      fb[ks][j] = *reinterpret_cast<const u32x4 *>(
          aw + off + (kTileN * sub + gemm_col<T>(wn, j, lr) - lr) * L::ROWB);
    }
  };
  // publish: every LDS read issued so far stays above the wait (the empty
  // asm pins memory accesses in program order)
  auto publish_step = [&]() {
    asm volatile("" ::: "memory");
    if (more)
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(kAhead, 0));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(kAhead - (STAGES - 2), 0));
    __builtin_amdgcn_s_barrier();
  };
  int cur = 0;  // buffer of slab s
  auto step = [&](int s, const FragA &fa, const FragB &fb, FragA &na, FragB &nb) {
    const int nxt = cur + 1 == STAGES ? 0 : cur + 1;
    publish_step();
    // the first kLead MFMAs of slab s go out right after the barrier, so
    // the matrix core restarts at once
#pragma unroll
    for (int idx = 0; idx < kLead; ++idx) {
      const int ks = idx / (T::FM * T::FN), i = (idx / T::FN) % T::FM, j = idx % T::FN;
      acc[i][j] = mfma_16x16x32_bf16(fa[ks][i], fb[ks][j], acc[i][j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    // the rest of the step in D chunks, each opening with one load
    // instruction of slab s + STAGES, then its share of slab s's MFMAs
    // interleaved with its share of slab s + 1's fragment reads
    const int slab_next = min(s + STAGES, slabs - 1);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      const int m0 = kLead + c * kRest / D, m1 = kLead + (c + 1) * kRest / D;
      const int r0 = c * kReads / D, r1 = (c + 1) * kReads / D;
      ring_load_one(slab_next, cur, c);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int idx = m0; idx < m1; ++idx) {
        const int ks = idx / (T::FM * T::FN), i = (idx / T::FN) % T::FM, j = idx % T::FN;
        acc[i][j] = mfma_16x16x32_bf16(fa[ks][i], fb[ks][j], acc[i][j]);
      }
#pragma unroll
      for (int r = r0; r < r1; ++r) read_frag(nxt, r, na, nb);
      // MFMA, read, MFMA, read, ..., then the chunk's remaining MFMAs
#pragma unroll
      for (int r = r0; r < r1; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
#pragma unroll
      for (int k = 0; k < (m1 - m0) - (r1 - r0); ++k)
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = nxt;
  };
#pragma unroll
  for (int p = 0; p < STAGES; ++p) ring_load(min(p, slabs - 1), p);
  FragA fa0, fa1;
  FragB fb0, fb1;
  if (more)
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(kAheadFirst, 0));
  else
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(kAheadFirst - (STAGES - 1), 0));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int r = 0; r < kReads; ++r) read_frag(0, r, fa0, fb0);
  int s = 0;
  for (; s + 2 <= slabs; s += 2) {
    step(s, fa0, fb0, fa1, fb1);
    step(s + 1, fa1, fb1, fa0, fb0);
  }
  if (s < slabs) step(s, fa0, fb0, fa1, fb1);
  // every load landed and every LDS read done before the ring is reused
  // for the staged tile (or the workgroup leaves)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(kWaitAll);
  if (EPI != kGemmF32 && a.vec_out) {
    __builtin_amdgcn_s_barrier();  // every wave's loads landed, ring read
    gemm_epilogue_staged<EPI, T>(a, tm, tn * T::NSUB + sub, wm, wn, lane, sw, acc,
                                 sb0 + sub * (kTileN * T::STAGE_COL));
  } else {
    gemm_epilogue<EPI, T>(a, tm, tn * T::NSUB + sub, wm, wn, lane, acc);
  }
}

// The same for a 256 x 256 tile (GemmTileWide): 64-deep slabs, so that a
// load instruction reads 128-byte row segments, in two buffers.  Three slabs
// of 64 KiB do not fit the LDS, and 32-deep ones, which did, read 64-byte
// segments: the load path then moves 46 GB/s a CU where 128-byte and longer
// ones reach 59 (256 x 256 tiles' loads alone, 32 CUs of an XCD on 4 x 8
// tiles; ring depths 3 to 5 alike), and the loads took longer than the
// products.  A slab comes in four units of 128 rows: A0, A1 (each wave row's
// first and last 64 of its 128 rows) and B0, B1 (fragment columns j < 2 and
// j >= 2).  Its 64 products a wave take two steps:
//   step 2s      A0 x B0, A0 x B1   while B1 and A1 of slab s are read
//   step 2s + 1  A1 x B1, A1 x B0   while A0 and B0 of slab s + 1 are read
// Each step opens with a wait and a barrier, which publish the units it
// reads and free those the step before read; these take the same units of
// slab s + 2: A0, B0 in step 2s, B1, A1 in step 2s + 1.  So every load has
// three steps to land (4 instructions a wave and step, 8 in flight past each
// wait) and two buffers hold what three would.  B0 of slab s + 1 is read
// over B1's registers: the two B register sets swap roles from slab to slab.
// K is added in the order of every other tile, bit for bit.
template <int EPI>
__device__ __forceinline__ void gemm_wide_run(const GemmArgs &a, int tm, int tn, uint16_t *sb0) {
  using T = GemmTileWide;
  constexpr int BK = kTileK;
  using L = DmaSlab<BK>;
  static_assert(T::FM == 8 && T::FN == 4 && T::BM == 256 && T::BN == 256, "unit geometry");
  constexpr int XB = T::BM * BK, kSlab = (T::BM + T::BN) * BK;  // bf16 elements
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int sub = wave / T::SUBWAVES;
  const int sw = wave % T::SUBWAVES;
  const int wm = sw / T::WN;
  const int wn = sw % T::WN;
  const int lr = lane & 15;
  const int g4 = lane >> 4;
  const int64_t k_bytes = a.k * 2;
  const u32x4 xw = buffer_rsrc_words(a.x, a.m * k_bytes);
  // the matrices of the tile's weight rows and its first row in each: gate
  // and up (SwiGLU), or of each sub-tile's head (q|k|v)
  u32x4 ww0, ww1;
  int64_t wrow0, wrow1;
  if constexpr (EPI == kGemmQkvRope) {
    const HeadRows h0 = head_rows(a, static_cast<int64_t>(tn) * 2);
    const HeadRows h1 = head_rows(a, static_cast<int64_t>(tn) * 2 + 1);
    ww0 = buffer_rsrc_words(h0.base, h0.rows * k_bytes);
    ww1 = buffer_rsrc_words(h1.base, h1.rows * k_bytes);
    wrow0 = h0.row;
    wrow1 = h1.row;
  } else {
    ww0 = buffer_rsrc_words(a.w0, a.n0 * k_bytes);
    ww1 = buffer_rsrc_words(EPI == kGemmSwiglu ? a.w1 : a.w0, a.n0 * k_bytes);
    wrow0 = wrow1 =
        static_cast<int64_t>(tn) * (EPI == kGemmSwiglu ? T::NSUB * kGemmHalfHead : T::BN);
  }

  // load instruction i (0 .. 15) of a unit fills its 8 rows 8 i ..; the
  // wave issues i = 2 wave + e, whose parity is e
  const int ld_r = lane / L::CH;
  int ld_off[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int f = ((L::RPI * e + ld_r) / L::RPB) % L::CH;
    ld_off[e] = ld_r * static_cast<int>(k_bytes) + 16 * ((lane % L::CH) ^ f);
  }
  const int fl = (lr / L::RPB) % L::CH;
  const int rd_off0 = lr * L::ROWB + 16 * (g4 ^ fl);
  const int rd_off1 = lr * L::ROWB + 16 * ((4 + g4) ^ fl);
  const int slabs = static_cast<int>(a.k / BK);
  const uint32_t ring_lds = lds_address(sb0);

  // row of the tile's 256 that row r (0 .. 127) of half `half` is
  auto unit_row = [](int r, int half) { return r % 64 + 128 * (r / 64) + 64 * half; };
  // h 0, 1: this wave's instructions of unit A<half>; 2, 3: of unit B<half>
  auto load_one = [&](int slab, int buf, int half, int h) __attribute__((always_inline)) {
    const int e = h & 1;
    const int trow = unit_row(L::RPI * (2 * wave + e), half);
    const int kb = slab * BK * 2;
    const uint32_t dst = ring_lds + static_cast<uint32_t>(buf * kSlab * 2 + trow * L::ROWB);
    if (h < 2) {
      const int64_t row = static_cast<int64_t>(tm) * T::BM + trow;
      dma_lds16(xw, ld_off[e] + static_cast<int>(row * k_bytes) + kb, dst);
    } else {
      // SwiGLU: sub-tile trow / 128 holds 64 gate rows (B0), 64 up rows (B1)
      const int64_t row =
          EPI == kGemmSwiglu
              ? wrow0 + (trow / kTileN) * kGemmHalfHead + trow % kGemmHalfHead
          : EPI == kGemmQkvRope ? (trow >= kTileN ? wrow1 : wrow0) + trow % kTileN
                                : wrow0 + trow;
      const bool second = EPI == kGemmQkvRope ? trow >= kTileN : half == 1;
      dma_lds16(second ? ww1 : ww0, ld_off[e] + static_cast<int>(row * k_bytes) + kb,
                dst + XB * 2);
    }
  };

  f32x4 acc[T::FM][T::FN];
#pragma unroll
  for (int i = 0; i < T::FM; ++i)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  using Quad = u32x4[2][4];  // [32-deep half][fragment] of an A unit
  using Pair = u32x4[2][2];  // of a B unit
  Quad fa0, fa1;
  Pair fb0, fb1;
  auto read_a = [&](int buf, int half, int r, Quad &f) __attribute__((always_inline)) {
    const int ks = r / 4, i = r % 4;
    f[ks][i] = *reinterpret_cast<const u32x4 *>(
        reinterpret_cast<const char *>(sb0 + buf * kSlab) + (ks ? rd_off1 : rd_off0) +
        (128 * wm + 64 * half + 16 * i) * L::ROWB);
  };
  auto read_b = [&](int buf, int half, int r, Pair &f) __attribute__((always_inline)) {
    const int ks = r / 2, j = r % 2;
    f[ks][j] = *reinterpret_cast<const u32x4 *>(
        reinterpret_cast<const char *>(sb0 + buf * kSlab + XB) + (ks ? rd_off1 : rd_off0) +
        (kTileN * sub + gemm_col<T>(wn, 2 * half + j, lr) - lr) * L::ROWB);
  };
  constexpr int kWaitStep = waitcnt_imm(8, 0);
  // One step: the 32 products of A unit `ha` (fragments `a_frag`) with B unit
  // `hb` (`b_first`), then with the other one (`b_second`), in 4 chunks of a
  // load instruction, 8 products and 3 fragment reads; loads(h) issues load
  // h, reads(r) makes fragment read r (0 .. 11).
  auto step = [&](const Quad &fa, int ha, const Pair &b_first, int hb, const Pair &b_second,
                  auto loads, auto reads) __attribute__((always_inline)) {
    auto product = [&](int idx) __attribute__((always_inline)) {
      const int half = idx / 16, ks = (idx / 8) % 2, i = (idx / 2) % 4, j = idx % 2;
      const int col = 2 * (half ? 1 - hb : hb) + j;
      const u32x4 b = half ? b_second[ks][j] : b_first[ks][j];
      acc[4 * ha + i][col] = mfma_16x16x32_bf16(fa[ks][i], b, acc[4 * ha + i][col]);
    };
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(kWaitStep);
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int idx = 0; idx < 4; ++idx) product(idx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      loads(c);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int idx = 4 + 7 * c; idx < 11 + 7 * c; ++idx) product(idx);
#pragma unroll
      for (int r = 3 * c; r < 3 * c + 3; ++r) reads(r);
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // both steps of a slab in buffer buf; b0 holds its B0 fragments on entry,
  // b1 those of slab s + 1 on return
  auto slab_steps = [&](int s, int buf, Pair &b0, Pair &b1) __attribute__((always_inline)) {
    const int next = min(s + 2, slabs - 1);
    step(fa0, 0, b0, 0, b1,
         [&](int h) __attribute__((always_inline)) { load_one(next, buf, 0, h); },
         [&](int r) __attribute__((always_inline)) {
           if (r < 4) read_b(buf, 1, r, b1);
           else read_a(buf, 1, r - 4, fa1);
         });
    step(fa1, 1, b1, 1, b0,
         [&](int h) __attribute__((always_inline)) { load_one(next, buf, 1, h); },
         [&](int r) __attribute__((always_inline)) {
           if (r < 8) read_a(1 - buf, 0, r, fa0);
           else read_b(1 - buf, 0, r - 8, b1);
         });
  };
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int h = 0; h < 4; ++h) load_one(min(p, slabs - 1), p, half, h);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(12, 0));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int r = 0; r < 8; ++r) read_a(0, 0, r, fa0);
#pragma unroll
  for (int r = 0; r < 4; ++r) read_b(0, 0, r, fb0);
  int s = 0;
  for (; s + 2 <= slabs; s += 2) {
    slab_steps(s, 0, fb0, fb1);
    slab_steps(s + 1, 1, fb1, fb0);
  }
  if (s < slabs) slab_steps(s, 0, fb0, fb1);
  // every load landed and every LDS read done before the ring is reused
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  if (EPI != kGemmF32 && a.vec_out) {
    __builtin_amdgcn_s_barrier();
    gemm_epilogue_staged<EPI, T>(a, tm, tn * T::NSUB + sub, wm, wn, lane, sw, acc,
                                 sb0 + sub * (kTileN * T::STAGE_COL));
  } else {
    gemm_epilogue<EPI, T>(a, tm, tn * T::NSUB + sub, wm, wn, lane, acc);
  }
}

// One launch covers the output with tiles of shape T and, when the last
// round of T tiles would leave at least half of the CUs idle, the last
// tail_n tile columns with tiles of half the height (TH, the same wave
// count): those columns then take one round of half tiles instead of a
// partial round of full ones (M = 2048, fused gate|up: 768 full tiles in 3
// rounds of 256, then 256 half tiles, instead of 3.5 rounds of full tiles).
// Workgroup b runs on XCD b % 8 (see "Tile order"); each XCD takes a
// contiguous range of full tiles first, then of half tiles, so the half
// tiles are dispatched last on every XCD.
template <int EPI, class T, int STAGES, class TH, int STAGES_H, int BK>
__global__ __launch_bounds__(T::WAVES *kWave) void gemm_kernel(GemmArgs a) {
  static_assert(TH::WAVES == T::WAVES, "one workgroup size");
  constexpr int kLds = GemmRing<T, STAGES, BK>::LDS > GemmRing<TH, STAGES_H, BK>::LDS
                           ? GemmRing<T, STAGES, BK>::LDS
                           : GemmRing<TH, STAGES_H, BK>::LDS;
  static_assert(kLds * 2 <= 160 * 1024, "LDS of one CU");
  __shared__ __attribute__((aligned(16))) uint16_t sb0[kLds];
  if constexpr (EPI == kGemmF32) {
    if (a.split_slabs) a.yf += static_cast<int64_t>(blockIdx.y) * a.split_stride;
  }
  const int xcd = static_cast<int>(blockIdx.x % kXcds);
  const int j = static_cast<int>(blockIdx.x / kXcds);
  int tm, tn;
  // padding workgroups leave as a whole: no barrier is skipped
  if (j < a.per_xcd) {
    if (!gemm_tile(xcd * a.per_xcd + j, a.tiles, a.tiles_m, a.tiles_n, tm, tn)) return;
    if constexpr (std::is_same<T, GemmTileWide>::value)
      gemm_wide_run<EPI>(a, tm, tn, sb0);
    else
      gemm_tile_run<EPI, T, STAGES, BK>(a, tm, tn, sb0);
    return;
  }
  if constexpr (!std::is_same<T, TH>::value) {
    if (!gemm_tile(xcd * a.hper_xcd + (j - a.per_xcd), a.htiles, a.htiles_m, a.htiles_n,
                   tm, tn))
      return;
    gemm_tile_run<EPI, TH, STAGES_H, BK>(a, tm, a.tiles_n + tn, sb0);
  }
}

// CUs of the device a stream runs on (cached per device; 256 on MI355X).
int gemm_device_cus(hipStream_t s) {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cached[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  if (s != nullptr) {
    hipDevice_t owner = 0;
    if (hipStreamGetDevice(s, &owner) != hipSuccess) return 256;
    dev = static_cast<int>(owner);
  }
  if (dev < 0 || dev >= kMaxDevices) return 256;
  int cus = cached[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
      cus = 256;
    cached[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

template <int EPI, int BK, class T, int STAGES, class TH = T, int STAGES_H = STAGES>
static hipError_t launch_tiles(GemmArgs &a, int64_t tiles_n, int cus, hipStream_t s,
                               int splits = 1) {
  const int64_t tiles_m = (a.m + T::BM - 1) / T::BM;
  const int64_t htiles_m = (a.m + TH::BM - 1) / TH::BM;
  int64_t tail_n = 0;
  if (!std::is_same<T, TH>::value) {
    const int64_t tiles = tiles_m * tiles_n;
    const int64_t rem = tiles % cus;
    if (tiles > cus && rem > 0 && 2 * rem <= cus) {
      const int64_t cols = (rem + tiles_m - 1) / tiles_m;
      if (cols < tiles_n && cols * htiles_m <= cus) tail_n = cols;
    }
  }
  const int64_t tiles = tiles_m * (tiles_n - tail_n);
  const int64_t htiles = htiles_m * tail_n;
  if (tiles + htiles > (int64_t{1} << 30)) return static_cast<hipError_t>(CASCADE_ESHAPE);
  a.tiles_m = static_cast<int32_t>(tiles_m);
  a.tiles_n = static_cast<int32_t>(tiles_n - tail_n);
  a.tiles = static_cast<int32_t>(tiles);
  a.per_xcd = static_cast<int32_t>((tiles + kXcds - 1) / kXcds);
  a.htiles_m = static_cast<int32_t>(htiles_m);
  a.htiles_n = static_cast<int32_t>(tail_n);
  a.htiles = static_cast<int32_t>(htiles);
  a.hper_xcd = static_cast<int32_t>((htiles + kXcds - 1) / kXcds);
  // 16-byte output accesses need 16-byte aligned rows in every buffer the
  // epilogue touches; otherwise the element-wise epilogue runs
  auto ok16 = [](const void *p) { return p == nullptr || aligned16(p); };
  a.vec_out = (a.ldy % 8 == 0) && ok16(a.y) && ok16(a.aux) && ok16(a.rope_cos) &&
              ok16(a.rope_sin) && ok16(a.k_out) && ok16(a.v_out) &&
              (a.kv_head_stride % 8 == 0);
  const int64_t grid = static_cast<int64_t>(kXcds) * (a.per_xcd + a.hper_xcd);
  return launch_kernel(gemm_kernel<EPI, T, STAGES, TH, STAGES_H, BK>,
                       dim3(static_cast<unsigned>(grid), static_cast<unsigned>(splits)),
                       dim3(T::WAVES * kWave), 0, s, a);
}

// Schedule of launch_tiles in rounds: whole rounds of full tiles, then a
// round of half-height tiles (tail 1), a partial round of full tiles
// (tail 2) or nothing (tail 0).
struct TileRounds {
  int64_t full;
  int tail;
};
// A round of 160 x 256 tiles, in rounds of 256 x 128 tiles of the same K
// (K = 4096: 70 to 76 us).  A launch is bounded by what each CU's load path
// moves (about 60 GB/s of X and W rows), so a round costs its rows of both,
// and rows of padding cost as much as any: 160 rows waste fewer of them at
// 129 .. 160 rows (logits of 157 rows 222 -> 209 us), 257 .. 320 (gate|up
// 92.7 -> 76.0 at 320; logits 374 -> 313) and 513 .. 640 (gate|up of 613
// rows 151.8 -> 139.2).  192-row tiles' ring of 3 would not fit the LDS.
constexpr double kLowRound = 1.3;
static TileRounds tile_rounds(int64_t tiles_m, int64_t tiles_n, int64_t htiles_m, int cus) {
  const int64_t tiles = tiles_m * tiles_n;
  const int64_t rem = tiles % cus;
  if (rem == 0) return {tiles / cus, 0};
  if (tiles > cus && 2 * rem <= cus) {
    const int64_t cols = (rem + tiles_m - 1) / tiles_m;
    if (cols < tiles_n && cols * htiles_m <= cus) return {tiles / cus, 1};
  }
  return {tiles / cus, 2};
}

// Short prompts: the streaming kernel (gemm_stream.hip).  Else 256-row tiles
// when there are at least as many as CUs: 256
// columns wide where their schedule is shorter (below), else 128 wide (a
// partial last round runs as 128-row half tiles); else 128-row tiles (a
// partial last round as 64-row half tiles),
// unless there are fewer of those than CUs and 64-row tiles need no more
// than twice their rounds: then 64-row tiles (the K / V projections,
// N = 1024, at M = 2048).
template <int EPI>
static hipError_t launch_gemm(GemmArgs &a, int64_t tiles_n, hipStream_t s) {
  const int cus = gemm_device_cus(s);
  const int64_t n = EPI == kGemmQkvRope  ? a.n0 + a.n1 + a.n2
                    : EPI == kGemmSwiglu ? 2 * a.n0
                                         : a.n0;
  const StreamPlan sp = stream_plan(EPI, a.m, n, cus);
  if (sp.fm) return launch_stream(EPI, sp, a, s);
  const int64_t tiles256 = (a.m + 255) / 256 * tiles_n;
  if (a.m > 128 && tiles256 >= cus) {
    // 256 x 256 tiles read a third less X and W per product, which is what
    // bounds these launches.  The schedule of rounds decides, with round
    // costs measured at M = 2048 and 8192, K = 4096 (in rounds of 256 x 128
    // tiles, about 57 us each): a round of 256 x 256 tiles 1.7 (97 us), a
    // round of their 128 x 256 half-height tail tiles 1.15, a round of
    // 128 x 128 tail tiles 0.7.  So the fused gate|up (N = 2 x 14336) at
    // M = 2048 runs 3 rounds + a half-height round of 256 x 256 (358 us)
    // rather than 7 rounds of 256 x 128 tiles (400 us); o_proj and q keep
    // their one round of 256 x 128 (57 us).  SwiGLU and q|k|v need whole
    // pairs of 128-column gate / up groups or heads.
    const int64_t tm256 = (a.m + 255) / 256, tm128 = (a.m + 127) / 128;
    const int64_t wide_n = (tiles_n + 1) / 2;
    const TileRounds std_r = tile_rounds(tm256, tiles_n, tm128, cus);
    const TileRounds wide_r = tile_rounds(tm256, wide_n, tm128, cus);
    constexpr double kWideRound = 1.7;  // in rounds of 256 x 128 tiles
    constexpr double kWideHalfRound = 1.15;
    constexpr double kHalfRound = 0.7;
    const double std_t = static_cast<double>(std_r.full) +
                         (std_r.tail == 1 ? kHalfRound : std_r.tail == 2 ? 1.0 : 0.0);
    const double wide_t = kWideRound * static_cast<double>(wide_r.full) +
                          (wide_r.tail == 1 ? kWideHalfRound : wide_r.tail == 2 ? kWideRound : 0.0);
    constexpr bool kWholePairs = EPI == kGemmSwiglu || EPI == kGemmQkvRope;
    const double low_t = kLowRound * static_cast<double>(
        ((a.m + 159) / 160 * wide_n + cus - 1) / cus);
    if (low_t < std::min(std_t, wide_t) && (!kWholePairs || tiles_n % 2 == 0))
      return launch_tiles<EPI, kTileK, GemmTile160, 3>(a, wide_n, cus, s);
    if (wide_t < std_t && (!kWholePairs || tiles_n % 2 == 0))
      return launch_tiles<EPI, kTileK, GemmTileWide, 2, GemmTileWideHalf, 3>(a, wide_n, cus, s);
    return launch_tiles<EPI, kTileK, GemmTile256, 3, GemmTile128x8, 4>(a, tiles_n, cus, s);
  }
  const int64_t tiles128 = (a.m + 127) / 128 * tiles_n;
  // fewer than one round of 128-row tiles still wins where it takes half
  // the rounds of 64-row tiles (M = 192 / 256, N = 14336: 61.8 -> 39.1 /
  // 62.6 -> 45.1 us)
  const int64_t rounds64 = ((a.m + 63) / 64 * tiles_n + cus - 1) / cus;
  const int64_t rounds128 = (tiles128 + cus - 1) / cus;
  if (tiles128 < cus && 2 * rounds128 > rounds64)
    return launch_tiles<EPI, kTileK, GemmTile64, 6>(a, tiles_n, cus, s);
  return launch_tiles<EPI, kTileK, GemmTile128, 4, GemmTile64, 6>(a, tiles_n, cus, s);
}

// Shared argument checks: X [m, k], K a multiple of the 64-deep slab.
// Byte offsets of the slab loads are 32-bit: X and every W stay below 2 GiB.
constexpr int64_t kGemmMaxBytes = int64_t{1} << 31;

static int gemm_check_x(const void *x, int64_t m, int64_t k) {
  if (x == nullptr || m <= 0 || k <= 0 || m > (int64_t{1} << 24))
    return CASCADE_EINVAL;
  if (!aligned16(x)) return CASCADE_EALIGN;
  if (k % kTileK) return CASCADE_ESHAPE;
  if (m * k * 2 >= kGemmMaxBytes) return CASCADE_ESHAPE;
  return 0;
}

static int gemm_check_w(const void *w, int64_t n, int64_t granule, int64_t k) {
  if (w == nullptr || n <= 0) return CASCADE_EINVAL;
  if (!aligned16(w)) return CASCADE_EALIGN;
  if (n % granule) return CASCADE_ESHAPE;
  if (n * k * 2 >= kGemmMaxBytes) return CASCADE_ESHAPE;
  return 0;
}

}  // namespace cascade

using namespace cascade;

// Split K.  Where 256-row tiles would keep at most half of the CUs busy over a
// long K (K >= 8192; prompts of 17 to 1280 rows over N = 4096: down_proj), K
// is split over up to kSplitMax rows of workgroups, each writing an fp32
// partial tile into the caller's workspace; a second launch sums the partials
// in split order and applies the element-wise epilogue at the same rounding
// points as the one-pass tile (bf16(sum), then the residual add).  The
// partials associate the K sum differently from one pass, so a result may
// differ from the one-pass tile in the last bf16 place, within the same
// rounding bound.  Up to 256 rows the streaming kernel writes the partials
// where it has enough runs (stream_split_plan), past that 256 x 128 tiles, or
// 160 x 256 tiles where, at kLowRound a tile, their more numerous splits are
// shorter (down_proj: 320 rows 53.7 -> 50.1 us, 613 rows 86.6 -> 73.4, 768
// rows 104 -> 92; 1100 and 1280 rows, whose 160 tiles of 256 x 128 do not
// split, 192 -> 120 and 218 -> 127).  Over a short K (o_proj) one pass ends
// before a split launch and its reduction (M = 64: 13.8 against 15.2 us; M =
// 192 .. 1024: 22.0 .. 33.8 against 23.3 .. 42.8).
constexpr int kSplitMax = 8;
constexpr int kSplitMinSlabs = 8;  // 64-deep slabs per split, at least
// Of 160 x 256 tiles: their ramp and the reduction of twice the partials
// outweigh shorter runs (N = 4096, 304 rows, 8 splits against 4 of 256 x 128
// tiles: K = 8192 43.8 and 36.9 us, 10240 47.7 and 42.5, 14336 50.2 and 54.5);
// nor does a split pay where one pass is a single round of 128-row tiles
// (N = 6144, K = 8192: 600 rows 75.7 us, one pass 68.9; 700 rows 78 and 110).
constexpr int kLowMinSlabs = 28;
constexpr int64_t kSplitMinK = 8192;

struct SplitPlan {
  int splits;  // 1: no split
  int per;     // slabs per split
  StreamPlan stream;  // fm: the streaming kernel writes the partials
  bool low;           // 160 x 256 tiles write them
};

static SplitPlan split_plan(int64_t m, int64_t n, int64_t k, int cus, bool low_tiles = true) {
  SplitPlan p{1, 0, {0, 0, 1}, false};
  // 16 rows and fewer: one pass streams the weight faster (M = 6,
  // down_proj: 23.3 us one pass, 21 + 4.7 split)
  if (m <= 16 || n % 8 != 0 || k % kTileK != 0 || k < kSplitMinK) return p;
  const int64_t slabs = k / kTileK;
  auto runs = [&](int64_t tiles) {
    return std::min<int64_t>(std::min<int64_t>(kSplitMax, cus / tiles), slabs / kSplitMinSlabs);
  };
  int64_t sp = runs((m + 255) / 256 * ((n + kTileN - 1) / kTileN));
  if (low_tiles && m > 256) {
    const int64_t low = runs((m + 159) / 160 * ((n + 255) / 256));
    const bool two_rounds = (m + 127) / 128 * ((n + kTileN - 1) / kTileN) > cus;
    p.low = low >= 2 && kLowRound * std::max<int64_t>(sp, 1) < low &&
            slabs >= kLowMinSlabs * low && (sp >= 2 || two_rounds);
    if (p.low) sp = low;
  }
  if (sp < 2) return p;
  p.stream = stream_split_plan(m, n, k, cus);
  if (p.stream.fm) sp = p.stream.splits;
  const int64_t per = (slabs + sp - 1) / sp;
  p.splits = static_cast<int>((slabs + per - 1) / per);  // no empty split
  p.stream.splits = p.splits;
  p.per = static_cast<int>(per);
  return p;
}

// y = epilogue(sum over s < splits of part[s]), 8 consecutive outputs per
// thread (n % 8 == 0, so a group never crosses a row).
template <int EPI>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(GemmArgs a, int splits) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (i >= a.m * a.n0) return;
  const float *p = a.yf + i;
  f32x4 lo = *reinterpret_cast<const f32x4 *>(p);
  f32x4 hi = *reinterpret_cast<const f32x4 *>(p + 4);
  for (int sp = 1; sp < splits; ++sp) {
    p += a.split_stride;
    lo += *reinterpret_cast<const f32x4 *>(p);
    hi += *reinterpret_cast<const f32x4 *>(p + 4);
  }
  const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  u32x4 aux = u32x4{0u, 0u, 0u, 0u};
  if constexpr (EPI == kGemmResidual) aux = *reinterpret_cast<const u32x4 *>(a.aux + i);
  u32x4 out;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float v0 = round_bf16(v[2 * q]), v1 = round_bf16(v[2 * q + 1]);
    if constexpr (EPI == kGemmResidual) {
      v0 = lo_f(aux[q]) + v0;
      v1 = hi_f(aux[q]) + v1;
    }
    out[q] = pack_bf16x2(v0, v1);
  }
  *reinterpret_cast<u32x4 *>(a.y + i) = out;
}

template <int EPI>
static int gemm_split_k(const GemmArgs &a, const SplitPlan &p, void *ws,
                        size_t ws_bytes, hipStream_t s) {
  static_assert(EPI == kGemmStore || EPI == kGemmResidual, "element-wise epilogues");
  const int64_t part = a.m * a.n0;
  if (ws_bytes < static_cast<size_t>(p.splits) * part * sizeof(float))
    return CASCADE_EWORKSPACE;
  GemmArgs b = a;
  b.yf = static_cast<float *>(ws);
  b.ldy = a.n0;
  b.split_slabs = p.per;
  b.split_stride = part;
  const int cus = gemm_device_cus(s);
  hipError_t e =
      p.stream.fm ? launch_stream(kGemmF32, p.stream, b, s)
      : p.low     ? launch_tiles<kGemmF32, kTileK, GemmTile160, 3>(b, (a.n0 + 255) / 256, cus, s,
                                                                   p.splits)
                  : launch_tiles<kGemmF32, kTileK, GemmTile256, 3>(
                        b, (a.n0 + kTileN - 1) / kTileN, cus, s, p.splits);
  if (e != hipSuccess) return e;
  GemmArgs r = a;
  r.yf = static_cast<float *>(ws);
  r.split_stride = part;
  const int64_t groups = (part / 8 + 255) / 256;
  return launch_kernel(gemm_split_reduce_kernel<EPI>, dim3(static_cast<unsigned>(groups)),
                       dim3(256), 0, s, r, p.splits);
}

static int gemm_plain(int epi, const void *x, const void *w, const void *aux,
                      void *y, int64_t m, int64_t n, int64_t k, void *stream) {
  if (int e = gemm_check_x(x, m, k)) return e;
  if (int e = gemm_check_w(w, n, 1, k)) return e;
  if (y == nullptr) return CASCADE_EINVAL;
  if (!aligned16(y)) return CASCADE_EALIGN;
  if ((epi == kGemmResidual || epi == kGemmMul) && aux == nullptr)
    return CASCADE_EINVAL;
  GemmArgs a{};
  a.x = static_cast<const uint16_t *>(x);
  a.w0 = static_cast<const uint16_t *>(w);
  a.n0 = n;
  a.m = m;
  a.k = k;
  a.y = static_cast<uint16_t *>(y);
  a.yf = static_cast<float *>(y);
  a.ldy = n;
  a.aux = static_cast<const uint16_t *>(aux);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t tiles_n = (n + kTileN - 1) / kTileN;
  switch (epi) {
    case kGemmStore: return launch_gemm<kGemmStore>(a, tiles_n, s);
    case kGemmResidual: return launch_gemm<kGemmResidual>(a, tiles_n, s);
    case kGemmSilu: return launch_gemm<kGemmSilu>(a, tiles_n, s);
    case kGemmMul: return launch_gemm<kGemmMul>(a, tiles_n, s);
    default: return launch_gemm<kGemmF32>(a, tiles_n, s);
  }
}

extern "C" int cascade_gemm_bf16(const void *x, const void *w, void *y,
                                 int64_t m, int64_t n, int64_t k,
                                 void *stream) {
  return gemm_plain(kGemmStore, x, w, nullptr, y, m, n, k, stream);
}

extern "C" int cascade_gemm_f32out_bf16(const void *x, const void *w,
                                        float *y, int64_t m, int64_t n,
                                        int64_t k, void *stream) {
  return gemm_plain(kGemmF32, x, w, nullptr, y, m, n, k, stream);
}

extern "C" int cascade_gemm_residual_bf16(const void *x, const void *w,
                                          const void *residual, void *y,
                                          int64_t m, int64_t n, int64_t k,
                                          void *stream) {
  return gemm_plain(kGemmResidual, x, w, residual, y, m, n, k, stream);
}

// The workspace forms: split K where the plan above applies (the workspace
// then needs cascade_gemm_workspace_bytes() bytes), else the one-pass GEMM.
static int gemm_ws(int epi, const void *x, const void *w, const void *aux,
                   void *y, int64_t m, int64_t n, int64_t k, void *workspace,
                   size_t workspace_bytes, void *stream) {
  if (int e = gemm_check_x(x, m, k)) return e;
  if (int e = gemm_check_w(w, n, 1, k)) return e;
  hipStream_t s = static_cast<hipStream_t>(stream);
  SplitPlan p = split_plan(m, n, k, gemm_device_cus(s));
  // where only the 160-row tiles split, a call without their workspace, or
  // whose workspace or residual is not 16-byte aligned, runs the one pass
  if (p.low && (workspace == nullptr || !aligned16(workspace) ||
                (aux != nullptr && !aligned16(aux)) ||
                workspace_bytes < static_cast<size_t>(p.splits) * m * n * sizeof(float))) {
    const SplitPlan one = split_plan(m, n, k, gemm_device_cus(s), false);
    if (one.splits == 1) p = one;
  }
  if (p.splits == 1)
    return gemm_plain(epi, x, w, aux, y, m, n, k, stream);
  if (y == nullptr || workspace == nullptr || (epi == kGemmResidual && aux == nullptr))
    return CASCADE_EINVAL;
  if (!aligned16(y) || !aligned16(workspace) || (aux != nullptr && !aligned16(aux)))
    return CASCADE_EALIGN;
  GemmArgs a{};
  a.x = static_cast<const uint16_t *>(x);
  a.w0 = static_cast<const uint16_t *>(w);
  a.n0 = n;
  a.m = m;
  a.k = k;
  a.y = static_cast<uint16_t *>(y);
  a.ldy = n;
  a.aux = static_cast<const uint16_t *>(aux);
  return epi == kGemmResidual
             ? gemm_split_k<kGemmResidual>(a, p, workspace, workspace_bytes, s)
             : gemm_split_k<kGemmStore>(a, p, workspace, workspace_bytes, s);
}

extern "C" size_t cascade_gemm_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0) return 0;
  const SplitPlan p = split_plan(m, n, k, gemm_device_cus(nullptr));
  return p.splits > 1 ? static_cast<size_t>(p.splits) * m * n * sizeof(float) : 0;
}

extern "C" int cascade_gemm_ws_bf16(const void *x, const void *w, void *y,
                                    int64_t m, int64_t n, int64_t k,
                                    void *workspace, size_t workspace_bytes,
                                    void *stream) {
  return gemm_ws(kGemmStore, x, w, nullptr, y, m, n, k, workspace,
                 workspace_bytes, stream);
}

extern "C" int cascade_gemm_residual_ws_bf16(const void *x, const void *w,
                                             const void *residual, void *y,
                                             int64_t m, int64_t n, int64_t k,
                                             void *workspace,
                                             size_t workspace_bytes,
                                             void *stream) {
  return gemm_ws(kGemmResidual, x, w, residual, y, m, n, k, workspace,
                 workspace_bytes, stream);
}

extern "C" int cascade_gate_silu_gemm_bf16(const void *x, const void *w_gate,
                                           void *y, int64_t m, int64_t n,
                                           int64_t k, void *stream) {
  return gemm_plain(kGemmSilu, x, w_gate, nullptr, y, m, n, k, stream);
}

extern "C" int cascade_up_mul_gemm_bf16(const void *x, const void *w_up,
                                        const void *gate, void *y, int64_t m,
                                        int64_t n, int64_t k, void *stream) {
  return gemm_plain(kGemmMul, x, w_up, gate, y, m, n, k, stream);
}

extern "C" int cascade_gate_up_swiglu_gemm_bf16(const void *x,
                                                const void *w_gate,
                                                const void *w_up, void *y,
                                                int64_t m, int64_t n_half,
                                                int64_t k, void *stream) {
  if (int e = gemm_check_x(x, m, k)) return e;
  if (int e = gemm_check_w(w_gate, n_half, kGemmHalfHead, k)) return e;
  if (int e = gemm_check_w(w_up, n_half, kGemmHalfHead, k)) return e;
  if (y == nullptr) return CASCADE_EINVAL;
  if (!aligned16(y)) return CASCADE_EALIGN;
  GemmArgs a{};
  a.x = static_cast<const uint16_t *>(x);
  a.w0 = static_cast<const uint16_t *>(w_gate);
  a.w1 = static_cast<const uint16_t *>(w_up);
  a.n0 = n_half;
  a.m = m;
  a.k = k;
  a.y = static_cast<uint16_t *>(y);
  a.ldy = n_half;
  return launch_gemm<kGemmSwiglu>(a, n_half / kGemmHalfHead,
                                  static_cast<hipStream_t>(stream));
}

extern "C" int cascade_qkv_rope_gemm_bf16(
    const void *x, int64_t m, const void *wq, const void *wk, const void *wv,
    int64_t nq, int64_t nk, int64_t nv, int64_t k, const void *rope_cos,
    const void *rope_sin, int64_t rope_positions, int64_t pos0, void *q_out,
    void *k_out, void *v_out, int64_t kv_head_stride, int64_t slot0,
    void *stream) {
  if (int e = gemm_check_x(x, m, k)) return e;
  if (nq < 0 || nk < 0 || nv < 0 || nq + nk + nv == 0) return CASCADE_EINVAL;
  if (std::max(nq, std::max(nk, nv)) * k * 2 >= kGemmMaxBytes) return CASCADE_ESHAPE;
  if ((nq % kGemmHead) || (nk % kGemmHead) || (nv % kGemmHead))
    return CASCADE_ESHAPE;
  if (nq && (wq == nullptr || q_out == nullptr)) return CASCADE_EINVAL;
  if (nk && (wk == nullptr || k_out == nullptr)) return CASCADE_EINVAL;
  if (nv && (wv == nullptr || v_out == nullptr)) return CASCADE_EINVAL;
  if ((nq && (!aligned16(wq) || !aligned16(q_out))) ||
      (nk && (!aligned16(wk) || !aligned16(k_out))) ||
      (nv && (!aligned16(wv) || !aligned16(v_out))))
    return CASCADE_EALIGN;
  if (nq || nk) {
    // every row's position must have a cos / sin row
    if (rope_cos == nullptr || rope_sin == nullptr || pos0 < 0 ||
        pos0 + m > rope_positions)
      return CASCADE_EINVAL;
  }
  if (nk || nv) {
    // every row's slot must lie inside each KV head's span
    if (slot0 < 0 || kv_head_stride < (slot0 + m) * kGemmHead ||
        (kv_head_stride & 7))
      return CASCADE_EINVAL;
  }
  GemmArgs a{};
  a.x = static_cast<const uint16_t *>(x);
  a.w0 = static_cast<const uint16_t *>(wq);
  a.w1 = static_cast<const uint16_t *>(wk);
  a.w2 = static_cast<const uint16_t *>(wv);
  a.n0 = nq;
  a.n1 = nk;
  a.n2 = nv;
  a.m = m;
  a.k = k;
  a.y = static_cast<uint16_t *>(q_out);
  a.ldy = nq;
  a.rope_cos = static_cast<const uint16_t *>(rope_cos);
  a.rope_sin = static_cast<const uint16_t *>(rope_sin);
  a.pos0 = pos0;
  a.k_out = static_cast<uint16_t *>(k_out);
  a.v_out = static_cast<uint16_t *>(v_out);
  a.kv_head_stride = kv_head_stride;
  a.slot0 = slot0;
  return launch_gemm<kGemmQkvRope>(a, (nq + nk + nv) / kGemmHead,
                                   static_cast<hipStream_t>(stream));
}
