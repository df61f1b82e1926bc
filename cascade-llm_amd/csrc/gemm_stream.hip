// Streaming GEMM for short prompts (2 .. 256 token rows) on gfx950, every
// epilogue of the prefill family (gemm.hip lists them).
//
// So few rows make the weights nearly all of the work: the launch is bounded
// by reading them once from HBM (about 6.5 TB/s for a launch of this kind),
// then by what each CU takes in besides, since a CU's loads return in order
// and the X lines that hit its XCD's L2 queue with the weight lines that do
// not.  So one workgroup per CU owns a run of weight rows that divides the
// matrix over the CUs (112 of the 28672 gate and up rows, 24 of the 6144 q|k|v
// rows, 16 of o_proj's 4096: not a power of two, so these rounds are full;
// other widths take the next built count, at most twice their share: gate|up
// of 4096, M = 6: 15.1 us on 32 rows, 23.2 on 112; logits of 8192 17.6 on 32,
// 24.3 on 128) and walks all of K once: the ramp of a launch is paid once, and
// every token row is read once per workgroup.  Where the token rows would
// outweigh the weight rows, 2 or 4 workgroups on one XCD take a share of the
// tokens and twice or four times the weight rows each (stream_plan).
//
// K is walked in slabs through a ring of LDS buffers (buffer loads straight to
// LDS, up to 148 KB in flight; slab depth 64 to 512 so that a step moves 16 KB
// or more), nontemporal where one workgroup alone reads the rows.  Up to 16
// rows over few columns a launch is a chain of steps with little to load in
// each: 512-deep slabs halve them, and waves that would repeat another one's
// fragment leave the LDS alone (M = 6, N = 1024: 8.0 -> 6.8 us, N = 4096 10.0
// -> 9.5; without the nontemporal hint 0.5 to 1.0 us less over K = 2048, 2.9
// more over K = 14336).  Waves 0-3 multiply the even 32-deep chunks of K,
// waves 4-7 the odd ones, each into two sums in turn, so that no chain of fp32
// additions is longer than a quarter of K (error of a product against 64 bits,
// K = 4096: 1.9e-7 of its norm, with one sum a wave 2.7e-7, one chain 4.0e-7);
// a quarter holds the same chunks whatever the shape of the workgroup (of up
// to 128 tokens).  The halves meet in LDS as an fp32 tile, from which the
// epilogue takes 4 columns (or 4 RoPE pairs) of a token at a time.
//
// Wide SwiGLU launches and the logits of a whole vocabulary start each tile at
// another run of K: with every CU on the same columns of rows 8 KB apart the
// same few channels serve all of them (112 rows a CU, loads alone: 44.9 ->
// 36.2 us); the sums of those launches depend on the start, hence on the tile,
// within the same bound.  The runs differ between the tiles of one XCD (tile /
// 8): taken from the tile number itself they agree within an XCD (logits of 26
// rows: 259 us, 217 without any, 174 so).  It pays from about 48 weight rows a
// CU on (gate|up of 7168, M = 33: 27.8 -> 23.1 us; of 4096 16.4 -> 19.1).  The
// other kinds, and narrower logits, add in one order whatever their width, so
// that a product does not depend on the columns beside it, though it would
// shorten them too (14336 columns, M = 6: 24.8 -> 20.6 us).
//
// Weights are the A operand, tokens the B operand: a lane then holds 4
// consecutive weight rows, i.e. output columns, of one token.  8-row blocks
// of gate rows alternate with the same 8 up rows, 4-row blocks of dims d
// with d + 64, so a fragment holds whole SwiGLU and RoPE pairs.
//
// LDS slab: rows of RB bytes, weight rows then token rows; 16-byte chunk c of
// operand row r sits at c ^ (r % 16) (64-deep slabs: c ^ ((r / 2) % 8)), so
// the 16 rows of a fragment read fall in distinct banks.
//
// Measured, MI355X, rotating weights, against the kernels it replaced
// (per launch): M = 6 gate|up 51.2 -> 38.0 us, q|k|v 18.2 -> 12.1; M = 45
// gate|up 70.1 -> 39.5 (5.9 TB/s), q|k|v 23.1 -> 15.5, o_proj 16.8 -> 13.0,
// down_proj (4 runs of K) 31.3 -> 26.4 with the reduction; M = 157 gate|up
// 73.6 -> 59.2, q|k|v 28.7 -> 22.7, o_proj 27.9 -> 17.1, k / v 18 -> 10.7;
// M = 26 logits of 128256 rows 259 -> 168.
#include <algorithm>
#include <type_traits>

#include "gemm_common.h"

namespace cascade {

// FM fragments of 16 tokens and NR weight rows of a workgroup.
template <int FM, int NR>
struct StreamShape {
  static constexpr int WAVES = 8;
  static constexpr int MT = 16 * FM;          // token rows of a workgroup
  static constexpr int FN = (NR + 15) / 16;   // fragments of its weight rows
  static constexpr int ROWS = NR + MT;
  static constexpr int BK = ROWS >= 128 ? 64 : ROWS >= 64 ? 128 : ROWS > 32 ? 256 : 512;
  static constexpr int RB = 2 * BK;           // bytes of one row in a slab
  static constexpr int CH = BK / 8;           // 16-byte chunks of it
  static constexpr int RPI = 1024 / RB;       // rows per load instruction
  static constexpr int WI = NR / RPI;         // load instructions: weights
  static constexpr int NI = ROWS / RPI;       // and all
  static constexpr int PER = (NI + WAVES - 1) / WAVES;
  static constexpr int SLAB = ROWS * RB;
  // the logits of a whole vocabulary take several rounds of workgroups: two
  // of them share a CU where 3 slabs each fit, one loading while the other
  // starts or stores (M = 26: 174 -> 168 us, M = 64: 194 -> 187)
  static constexpr bool TWO = NR == 128 && 2 * 3 * SLAB <= 158000;
  static constexpr int FIT = (TWO ? 79000 : 151552) / SLAB;
  static constexpr int STAGES = BK == 512 ? 3 : FIT > 12 ? 12 : FIT;
  static constexpr int PITCH = 16 * FN + 4;   // floats per token of the staged tile
  static constexpr int LDS = std::max(STAGES * SLAB, MT * PITCH * 4);
  // 4 waves of each K half share the fragments
  static constexpr int WN = FN >= 4 && FM < 5 ? 4 : FN >= 2 ? 2 : 1;
  static constexpr int WM = 4 / WN;
  static constexpr int FMW = (FM + WM - 1) / WM;
  static constexpr int FNW = (FN + WN - 1) / WN;
  // sums of a fragment in a wave (160 tokens: one, half of K; the second cost
  // 0.6% of a layer of 157 rows)
  static constexpr int SUMS = FM <= 8 ? 2 : 1;
  static_assert(NR % 8 == 0 && STAGES >= 3 && LDS <= 160 * 1024, "shape");
  static_assert((STAGES - 1) * PER < 64, "vmcnt holds 6 bits");
};

// buffer_load ... lds with the nontemporal hint (weights read by one
// workgroup only), otherwise dma_lds16.
__device__ __forceinline__ void dma_lds16_nt(const u32x4 &rsrc, int voff, uint32_t lds) {
  u32x4 r;
  r.x = __builtin_amdgcn_readfirstlane(rsrc.x);
  r.y = __builtin_amdgcn_readfirstlane(rsrc.y);
  r.z = __builtin_amdgcn_readfirstlane(rsrc.z);
  r.w = __builtin_amdgcn_readfirstlane(rsrc.w);
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(r)
               : "memory", "m0");
}

template <int EPI, int FM, int NR>
__global__ __launch_bounds__(512) void gemm_stream_kernel(GemmArgs a) {
  using S = StreamShape<FM, NR>;
  constexpr bool kPairs = EPI == kGemmQkvRope || EPI == kGemmSwiglu;
  __shared__ __attribute__((aligned(16))) unsigned char ring[S::LDS];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lr = lane & 15;
  const int g4 = lane >> 4;
  const int tile = static_cast<int>(blockIdx.x);
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * S::MT;
  const int64_t k_bytes = a.k * 2;
  // this split's 64-deep pieces of K
  const int pieces = static_cast<int>(a.k / 64);
  const int piece0 = a.split_slabs ? static_cast<int>(blockIdx.z) * a.split_slabs : 0;
  const int count = a.split_slabs ? min(a.split_slabs, pieces - piece0) : pieces;
  const int slabs = (count * 64 + S::BK - 1) / S::BK;
  // (in runs of 256 columns of K, whatever the slab depth: the products of
  // a fused launch and of its halves then add in the same order; a K of an
  // odd number of 64-deep slabs would start the second round of them in the
  // other sum)
  const int rot = S::BK <= 256 && a.rotate && a.k >= 256 && a.k % 128 == 0
                      ? tile / kXcds % static_cast<int>(a.k / 256) * (256 / std::min(256, S::BK))
                      : 0;

  // load instruction t of this wave: wave + 8 t of the slab's NI (weight
  // rows, then token rows)
  const int ld_r = lane / S::CH;
  u32x4 rsrc[S::PER];
  int voff[S::PER];
#pragma unroll
  for (int t = 0; t < S::PER; ++t) {
    const int i = wave + S::WAVES * t;
    const int r = i * S::RPI + ld_r;  // slab row
    const uint16_t *base;
    int64_t rows, row;
    if (i >= S::WI) {
      base = a.x; rows = a.m; row = row0 + r - NR;
    } else if constexpr (EPI == kGemmSwiglu) {
      const bool up = (i * S::RPI) & 8;
      base = up ? a.w1 : a.w0;
      rows = a.n0;
      row = static_cast<int64_t>(tile) * (NR / 2) + 8 * (r / 16) + r % 8;
    } else if constexpr (EPI == kGemmQkvRope) {
      // rows 8 q + 0..3 / 4..7: dims d .. d + 3 / d + 64 .. of 4 pairs
      const int64_t pair = static_cast<int64_t>(tile) * (NR / 2) + 4 * ((i * S::RPI) / 8);
      const int64_t head = pair / kGemmHalfHead;
      const int64_t hq = a.n0 / kGemmHead, hk = a.n1 / kGemmHead;
      int64_t h = head;
      if (head < hq) {
        base = a.w0; rows = a.n0;
      } else if (head < hq + hk) {
        base = a.w1; rows = a.n1; h = head - hq;
      } else {
        base = a.w2; rows = a.n2; h = head - hq - hk;
      }
      row = h * kGemmHead + pair % kGemmHalfHead + r % 4 + (r % 8 >= 4 ? kGemmHalfHead : 0);
    } else {
      base = a.w0; rows = a.n0; row = static_cast<int64_t>(tile) * NR + r;
    }
    rsrc[t] = buffer_rsrc_words(base, rows * k_bytes);
    const int sr = i >= S::WI ? r - NR : r;  // row within its operand
    const int f = S::CH == 8 ? (sr / 2) % 8 : sr % 16;
    voff[t] = static_cast<int>(row * k_bytes) + 128 * piece0 + 16 * ((lane % S::CH) ^ f);
  }
  const bool stream_w = gridDim.y == 1 && (S::BK < 512 || a.k >= 4096);
  const uint32_t ring_lds = lds_address(ring);
  auto load_slab = [&](int slab, int buf) {
    int at = min(slab, slabs - 1) + rot;
    if (at >= slabs) at -= slabs;
    const uint32_t dst = ring_lds + static_cast<uint32_t>(buf * S::SLAB);
#pragma unroll
    for (int t = 0; t < S::PER; ++t) {
      const int i = wave + S::WAVES * t;
      if (S::NI % S::WAVES != 0 && t == S::PER - 1 && i >= S::NI) break;
      if (i < S::WI && stream_w)
        dma_lds16_nt(rsrc[t], voff[t] + at * S::RB, dst + i * 1024);
      else
        dma_lds16(rsrc[t], voff[t] + at * S::RB, dst + i * 1024);
    }
  };

  // K halves: 32-deep chunks of even / odd index; the 4 waves of a half
  // take fragments wn, wn + WN, .. of the weights and wm, wm + WM, .. of the
  // tokens (past the end: the last one again, not stored)
  const int kg = wave / 4;
  const int wn = wave % S::WN;
  const int wm = (wave % 4) / S::WN;
  // waves left without a fragment of their own only load
  const bool idle = S::WM >= 2 * FM && wm >= FM;
  f32x4 acc[S::SUMS][S::FMW][S::FNW];  // the half's chunks go to either sum in turn
#pragma unroll
  for (int e = 0; e < S::SUMS; ++e)
#pragma unroll
    for (int i = 0; i < S::FMW; ++i)
#pragma unroll
      for (int j = 0; j < S::FNW; ++j) acc[e][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int fl = S::CH == 8 ? (lr / 2) % 8 : lr;
  constexpr int KS = S::BK / 64;  // chunks of a wave's K half in a slab
  struct Frags {
    u32x4 w[KS][S::FNW], x[KS][S::FMW];
  };
  auto read_frags = [&](int buf, Frags &f) __attribute__((always_inline)) {
    if (idle) return;
    const unsigned char *b0 = ring + buf * S::SLAB + lr * S::RB;
#pragma unroll
    for (int q = 0; q < KS; ++q) {
      const int off = 16 * ((4 * (2 * q + kg) + g4) ^ fl);
#pragma unroll
      for (int j = 0; j < S::FNW; ++j)
        f.w[q][j] = *reinterpret_cast<const u32x4 *>(
            b0 + 16 * min(wn + S::WN * j, S::FN - 1) * S::RB + off);
#pragma unroll
      for (int i = 0; i < S::FMW; ++i)
        f.x[q][i] = *reinterpret_cast<const u32x4 *>(
            b0 + (NR + 16 * min(wm + S::WM * i, FM - 1)) * S::RB + off);
    }
  };
  // odd: an odd slab (64-deep slabs hold one chunk of the wave's half each)
  auto multiply = [&](int slab, const Frags &f, auto odd) __attribute__((always_inline)) {
    int at = slab + rot;
    if (at >= slabs) at -= slabs;
    const int valid = count * 2 - at * (S::BK / 32);  // 32-deep chunks left
    if (idle) return;
#pragma unroll
    for (int q = 0; q < KS; ++q) {
      if (KS > 1 && 2 * q + kg >= valid) break;
      constexpr int kOdd = decltype(odd)::value;
      const int set = S::SUMS == 1 ? 0 : KS == 1 ? kOdd : q & 1;
#pragma unroll
      for (int i = 0; i < S::FMW; ++i)
#pragma unroll
        for (int j = 0; j < S::FNW; ++j)
          acc[set][i][j] = mfma_16x16x32_bf16(f.w[q][j], f.x[q][i], acc[set][i][j]);
    }
  };
  // Slab s in ring buffer s % STAGES.  Step s waits for this wave's loads of
  // slab s + 1 and its LDS reads of slab s; one barrier publishes slab
  // s + 1 and frees slab s's buffer, which takes slab s + STAGES; slab
  // s + 1's fragments are read while slab s's products run.  Past the last
  // slab: the last one again, never used.
  const bool more = S::NI % S::WAVES == 0 || wave < S::NI % S::WAVES;
  auto publish = [&](auto ahead) __attribute__((always_inline)) {
    constexpr int kSlabs = decltype(ahead)::value;
    asm volatile("" ::: "memory");
    if (more)
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(kSlabs * S::PER, 0));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(kSlabs * (S::PER - 1), 0));
    __builtin_amdgcn_s_barrier();
  };
#pragma unroll
  for (int p = 0; p < S::STAGES; ++p) load_slab(p, p);
  Frags f0, f1;
  publish(std::integral_constant<int, S::STAGES - 1>{});
  read_frags(0, f0);
  int buf = 0;
  auto step = [&](int slab, const Frags &here, Frags &next, auto odd)
      __attribute__((always_inline)) {
    publish(std::integral_constant<int, S::STAGES - 2>{});
    load_slab(slab + S::STAGES, buf);
    buf = buf + 1 == S::STAGES ? 0 : buf + 1;
    read_frags(buf, next);
    multiply(slab, here, odd);
  };
  constexpr std::integral_constant<int, 0> kEven;
  constexpr std::integral_constant<int, 1> kOdd;
  int slab = 0;
  for (; slab + 2 <= slabs; slab += 2) {
    step(slab, f0, f1, kEven);
    step(slab + 1, f1, f0, kOdd);
  }
  if (slab < slabs) step(slab, f0, f1, kEven);
  // every load landed and every LDS read done before the ring holds the tile
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __syncthreads();
  if constexpr (S::SUMS == 2) {
#pragma unroll
    for (int i = 0; i < S::FMW; ++i)
#pragma unroll
      for (int j = 0; j < S::FNW; ++j) acc[0][i][j] += acc[1][i][j];
  }
  float *tile_f = reinterpret_cast<float *>(ring);
  auto each = [&](auto f) {
#pragma unroll
    for (int i = 0; i < S::FMW; ++i)
#pragma unroll
      for (int j = 0; j < S::FNW; ++j) {
        const int fi = wm + S::WM * i, fj = wn + S::WN * j;
        if (fi < FM && fj < S::FN)
          f(reinterpret_cast<f32x4 *>(tile_f + (16 * fi + lr) * S::PITCH + 16 * fj + 4 * g4),
            acc[0][i][j]);
      }
  };
  if (kg == 1) each([](f32x4 *p, const f32x4 &v) { *p = v; });
  __syncthreads();
  if (kg == 0) each([](f32x4 *p, const f32x4 &v) { *p = v + *p; });
  __syncthreads();

  // 4 consecutive output columns (or 4 RoPE pairs) of one token per item
  constexpr int kGroups = kPairs ? NR / 8 : NR / 4;
  const int tokens = static_cast<int>(min<int64_t>(S::MT, a.m - row0));
  for (int item = tid; item < tokens * kGroups; item += 512) {
    const int token = item / kGroups;
    const int g = item % kGroups;
    const int64_t row = row0 + token;
    const float *src = tile_f + token * S::PITCH;
    if constexpr (EPI == kGemmQkvRope) {
      const f32x4 lo = *reinterpret_cast<const f32x4 *>(src + 8 * g);
      const f32x4 hi = *reinterpret_cast<const f32x4 *>(src + 8 * g + 4);
      const int64_t pair = static_cast<int64_t>(tile) * (NR / 2) + 4 * g;
      const int64_t head = pair / kGemmHalfHead;
      const int d = static_cast<int>(pair % kGemmHalfHead);
      const int64_t hq = a.n0 / kGemmHead, hk = a.n1 / kGemmHead;
      if (head >= hq + hk + a.n2 / kGemmHead) continue;
      uint16_t ol[4], oh[4];
      if (head < hq + hk) {
        const uint16_t *cs = a.rope_cos + (a.pos0 + row) * kGemmHalfHead + d;
        const uint16_t *sn = a.rope_sin + (a.pos0 + row) * kGemmHalfHead + d;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float c = bf16_to_f32(cs[e]), s = bf16_to_f32(sn[e]);
          const float xa = round_bf16(lo[e]), xb = round_bf16(hi[e]);
          ol[e] = f32_to_bf16(round_bf16(xa * c) + round_bf16(-xb * s));
          oh[e] = f32_to_bf16(round_bf16(xb * c) + round_bf16(xa * s));
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ol[e] = f32_to_bf16(lo[e]);
          oh[e] = f32_to_bf16(hi[e]);
        }
      }
      uint16_t *dst;
      if (head < hq)
        dst = a.y + row * a.ldy + head * kGemmHead + d;
      else if (head < hq + hk)
        dst = a.k_out + (head - hq) * a.kv_head_stride + (a.slot0 + row) * kGemmHead + d;
      else
        dst = a.v_out + (head - hq - hk) * a.kv_head_stride + (a.slot0 + row) * kGemmHead + d;
      if (a.vec_out) {
        *reinterpret_cast<uint2 *>(dst) = *reinterpret_cast<const uint2 *>(ol);
        *reinterpret_cast<uint2 *>(dst + kGemmHalfHead) = *reinterpret_cast<const uint2 *>(oh);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          dst[e] = ol[e];
          dst[e + kGemmHalfHead] = oh[e];
        }
      }
    } else {
      const int64_t col = static_cast<int64_t>(tile) * (EPI == kGemmSwiglu ? NR / 2 : NR) + 4 * g;
      if (col >= a.n0) continue;
      const int64_t at = row * a.ldy + col;
      const bool vec = a.vec_out && col + 4 <= a.n0;
      if constexpr (EPI == kGemmF32) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(src + 4 * g);
        float *dst = a.yf + static_cast<int64_t>(blockIdx.z) * a.split_stride + at;
        if (vec) {
          *reinterpret_cast<f32x4 *>(dst) = v;
        } else {
          for (int e = 0; e < 4 && col + e < a.n0; ++e) dst[e] = v[e];
        }
      } else {
        float o[4];
        if constexpr (EPI == kGemmSwiglu) {
          const int r = 16 * (g / 2) + 4 * (g % 2);
          const f32x4 gt = *reinterpret_cast<const f32x4 *>(src + r);
          const f32x4 up = *reinterpret_cast<const f32x4 *>(src + r + 8);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = round_bf16(gemm_silu(round_bf16(gt[e]))) * round_bf16(up[e]);
        } else {
          const f32x4 v = *reinterpret_cast<const f32x4 *>(src + 4 * g);
          float aux[4] = {0.0f, 0.0f, 0.0f, 0.0f};
          if constexpr (EPI == kGemmResidual || EPI == kGemmMul) {
            if (vec) {
              const uint2 u = *reinterpret_cast<const uint2 *>(a.aux + at);
              aux[0] = lo_bf16(u.x); aux[1] = hi_bf16(u.x);
              aux[2] = lo_bf16(u.y); aux[3] = hi_bf16(u.y);
            } else {
              for (int e = 0; e < 4 && col + e < a.n0; ++e) aux[e] = bf16_to_f32(a.aux[at + e]);
            }
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float r = round_bf16(v[e]);
            if constexpr (EPI == kGemmResidual) o[e] = aux[e] + r;
            else if constexpr (EPI == kGemmSilu) o[e] = gemm_silu(r);
            else if constexpr (EPI == kGemmMul) o[e] = aux[e] * r;
            else o[e] = r;
          }
        }
        if (vec) {
          *reinterpret_cast<uint2 *>(a.y + at) =
              uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
        } else {
          for (int e = 0; e < 4 && col + e < a.n0; ++e) a.y[at + e] = f32_to_bf16(o[e]);
        }
      }
    }
  }
}

// ------------------------------------------------------------------ launch

template <int EPI, int FM, int NR>
static hipError_t launch_stream_shape(const GemmArgs &args, int64_t n, hipStream_t s,
                                      int splits = 1) {
  GemmArgs a = args;
  auto ok = [](const void *p, uintptr_t mask) {
    return (reinterpret_cast<uintptr_t>(p) & mask) == 0;
  };
  // 8-byte output accesses (16-byte for fp32)
  a.vec_out = a.ldy % 4 == 0 && ok(a.y, 7) && ok(a.yf, 15) && ok(a.aux, 7) && ok(a.k_out, 7) &&
              ok(a.v_out, 7) && a.kv_head_stride % 4 == 0;
  const int64_t tiles = (n + NR - 1) / NR;
  const int64_t mt = (a.m + 16 * FM - 1) / (16 * FM);
  if (tiles > 0x7fffffff || mt > 65535) return static_cast<hipError_t>(CASCADE_ESHAPE);
  // The workgroups that share a tile's weight rows run on one XCD, or each
  // reads them from memory again: up to 7 workgroups more in each row of
  // them, past every weight row (their loads read zeros, they store nothing),
  // while all fit the CUs.  (A test of the tile in the kernel made every
  // launch 0.2 us longer.)
  int64_t grid = (tiles + kXcds - 1) / kXcds * kXcds;
  if (mt == 1 || grid * mt * splits > gemm_device_cus(s)) grid = tiles;
  return launch_kernel(gemm_stream_kernel<EPI, FM, NR>,
                       dim3(static_cast<unsigned>(grid), static_cast<unsigned>(mt),
                            static_cast<unsigned>(splits)),
                       dim3(512), 0, s, a);
}

// Shapes a kind is built for: weight rows per workgroup (ascending) and the
// token fragments each is built for.
template <int... V>
struct Ints {};

// Those a plan can ask for.  Below 64 rows (of both matrices) the token tiles
// are as many as wanted (stream_plan), so that 4 fragments hold their share;
// 10 fragments come with more than 64, and for fp32 with partials of split K
// only (logits stop at 128 tokens).
constexpr bool stream_built(int epi, int rows, int fm) {
  if (epi == kGemmQkvRope) return true;
  const int all = epi == kGemmSilu || epi == kGemmMul ? 2 * rows : rows;
  if (all < 64) return fm <= 4;
  return fm < 10 || (all > 64 && (epi != kGemmF32 || rows == 128));
}

template <int EPI, int NR, int... FMS>
static hipError_t launch_fm(int fm, Ints<FMS...>, const GemmArgs &a, int64_t n, hipStream_t s,
                            int splits) {
  hipError_t e = static_cast<hipError_t>(CASCADE_ESHAPE);
  auto launch = [&](auto shape) {
    constexpr int kFm = decltype(shape)::value;
    if constexpr (stream_built(EPI, NR, kFm))
      e = launch_stream_shape<EPI, kFm, NR>(a, n, s, splits);
    return true;
  };
  (void)((fm == FMS && launch(std::integral_constant<int, FMS>{})) || ...);
  return e;
}

template <int EPI, class Fms, int... NRS>
static hipError_t launch_nr(int nr, int fm, Ints<NRS...>, const GemmArgs &a, int64_t n,
                            hipStream_t s, int splits) {
  hipError_t e = static_cast<hipError_t>(CASCADE_ESHAPE);
  (void)((nr == NRS ? (e = launch_fm<EPI, NRS>(fm, Fms{}, a, n, s, splits), true) : false) ||
         ...);
  return e;
}

using StreamFms = Ints<1, 2, 3, 4, 5, 6, 8, 10>;
using StreamFmsQkv = Ints<1, 2, 3, 4, 5>;
using StreamRows = Ints<16, 32, 64, 112>;              // plain, residual
using StreamRowsQkv = Ints<16, 24, 32, 48, 64, 96>;
using StreamRowsSwiglu = Ints<16, 32, 64, 112>;
using StreamRowsHalf = Ints<8, 16, 32, 56>;            // silu, mul: half of swiglu's
using StreamRowsF32 = Ints<16, 32, 64, 112, 128>;      // logits; split-K partials

template <int... V>
static int at_least(Ints<V...>, int64_t want) {  // smallest built value >= want, or 0
  int r = 0;
  (void)((V >= want ? (r = V, true) : false) || ...);
  return r;
}
template <int... V>
static int largest(Ints<V...>) {
  int r = 0;
  ((r = V), ...);
  return r;
}

static int rows_for(int epi, int64_t want) {
  auto pick = [&](auto list) {
    const int r = at_least(list, want);
    return r ? r : largest(list);
  };
  switch (epi) {
    case kGemmQkvRope: return pick(StreamRowsQkv{});
    case kGemmSwiglu: return pick(StreamRowsSwiglu{});
    case kGemmSilu:
    case kGemmMul: return pick(StreamRowsHalf{});
    case kGemmF32: return pick(StreamRowsF32{});
    default: return pick(StreamRows{});
  }
}

// Up to 256 rows over at most 24 weight rows a CU (q|k|v, o, k, v), 160 over
// more (gate|up at M = 157: 59.2 us against 73.6 on 128-row tiles), 128 for
// logits (M = 128: 230 us against 250 on 256 x 256 tiles; M = 157: 266
// against 250).  Past 128 rows over 32 to 64 weight rows a CU one round of
// tiles is shorter (M = 160: N = 10240 31.0 us, 35.0 here; 14336 36.6, 38.5;
// 20480, two rounds, 62.8, 51.3), except for q|k|v, whose launches a matrix
// at a time must add like the fused one.
// Token tiles by M, each measured best at N = 4096 / 6144 over
// K = 4096: one up to 48 rows (M = 45: 13.0 us, two 14.5), two up
// to 112 (M = 100: 15.0, one 18.2; q|k|v to 160: 22.7, four 23.4), then four
// (M = 157: 17.1, two 19.3); always one past 48 weight rows a CU, where the
// weights outweigh the tokens again (M = 64: N = 14336 28.0 us, two 31.6;
// N = 8192, M = 100: two 21.6, one 26.7).
StreamPlan stream_plan(int epi, int64_t m, int64_t n, int cus) {
  const StreamPlan none{0, 0, 1};
  const bool half = epi == kGemmSilu || epi == kGemmMul;
  const bool paired = epi == kGemmSwiglu || half;
  // weight rows of the launch, of a half those of both, so that the fused
  // launch and its halves take the same tiles
  const int64_t all = half ? 2 * n : n;
  if (m > (epi == kGemmF32 ? 128 : paired || all > 24 * static_cast<int64_t>(cus) ? 160 : 256))
    return none;
  if (m > 128 && epi != kGemmQkvRope && all > 32 * static_cast<int64_t>(cus) &&
      all <= 64 * static_cast<int64_t>(cus))
    return none;
  // token tiles wanted: the bytes a workgroup loads are its weight rows plus
  // its tokens' rows, least where the two are about equal
  const int64_t per_cu = (n + cus - 1) / cus;
  const int64_t want = m <= 48 || all > 48 * static_cast<int64_t>(cus) ? 1
                       : m <= (epi == kGemmQkvRope ? 160 : 112)        ? 2
                                                                       : 4;
  StreamPlan p;
  p.rows = rows_for(epi, per_cu * want);
  const int64_t tiles = (n + p.rows - 1) / p.rows;
  const int64_t frags = (m + 15) / 16;
  const int64_t mt = std::max<int64_t>(1, std::min(cus / tiles, frags));
  const int64_t fm = (frags + mt - 1) / mt;
  p.fm = epi == kGemmQkvRope ? at_least(StreamFmsQkv{}, fm) : at_least(StreamFms{}, fm);
  p.splits = 1;
  return p.fm && stream_built(epi, p.rows, p.fm) ? p : none;
}

// down_proj (K = 14336, N = 4096): in one pass each of 256 workgroups would
// read 28 KB of every token row for 16 weight rows (M = 45: 36.3 us); 64 weight
// rows over a quarter of K read 7 KB (22.9 us and 4.7 for the reduction).
// 128 rows over an eighth past 112 token rows (M = 100: 28.8 against 27.9 us,
// but twice the partials; M = 157: 37.5 against 32.9).  Over more columns
// fewer runs fit, and 256 x 128 tiles with twice as many end first: two runs
// of 64 rows past 64 token rows (8192 columns over K = 28672, M = 112: 111 us
// tiles, 120 here; M = 64: 100, 101), two or three past 160 (N = 5120, M = 200:
// 48, 54; N = 8192: 129, 156; four, N = 4096: 47.0, 45.5).
StreamPlan stream_split_plan(int64_t m, int64_t n, int64_t k, int cus) {
  StreamPlan p{0, 0, 1};
  if (m <= 16 || m > 256 || k < 8192) return p;
  p.rows = m <= 112 ? 64 : 128;
  const int64_t mt = m <= 160 ? 1 : 2;
  const int64_t tiles = (n + p.rows - 1) / p.rows * mt;
  const int64_t slabs = k / 64;
  const int64_t sp = std::min<int64_t>(std::min<int64_t>(8, cus / tiles), slabs / 8);
  if (sp < (m <= 64 ? 2 : m <= 160 ? 3 : 4)) return p;
  p.fm = at_least(StreamFms{}, ((m + 15) / 16 + mt - 1) / mt);
  p.splits = static_cast<int>(sp);
  return p;
}

hipError_t launch_stream(int epi, const StreamPlan &p, const GemmArgs &args, hipStream_t s) {
  GemmArgs a = args;
  const int64_t n = epi == kGemmQkvRope  ? a.n0 + a.n1 + a.n2
                    : epi == kGemmSwiglu ? 2 * a.n0
                                         : a.n0;
  if (epi == kGemmSwiglu || epi == kGemmSilu || epi == kGemmMul)
    a.rotate = 2 * a.n0 > 48 * static_cast<int64_t>(gemm_device_cus(s));
  else
    a.rotate = epi == kGemmF32 && p.splits == 1 && n > 65536;
  switch (epi) {
    case kGemmStore:
      return launch_nr<kGemmStore, StreamFms>(p.rows, p.fm, StreamRows{}, a, n, s, 1);
    case kGemmResidual:
      return launch_nr<kGemmResidual, StreamFms>(p.rows, p.fm, StreamRows{}, a, n, s, 1);
    case kGemmQkvRope:
      return launch_nr<kGemmQkvRope, StreamFmsQkv>(p.rows, p.fm, StreamRowsQkv{}, a, n, s, 1);
    case kGemmSwiglu:
      return launch_nr<kGemmSwiglu, StreamFms>(p.rows, p.fm, StreamRowsSwiglu{}, a, n, s, 1);
    case kGemmSilu:
      return launch_nr<kGemmSilu, StreamFms>(p.rows, p.fm, StreamRowsHalf{}, a, n, s, 1);
    case kGemmMul:
      return launch_nr<kGemmMul, StreamFms>(p.rows, p.fm, StreamRowsHalf{}, a, n, s, 1);
    default:
      return launch_nr<kGemmF32, StreamFms>(p.rows, p.fm, StreamRowsF32{}, a, n, s, p.splits);
  }
}

}  // namespace cascade
