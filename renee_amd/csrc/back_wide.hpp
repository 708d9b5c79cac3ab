// Both products of the backward pass and the update in one pass over the labels, as in back_step.hpp, for 257 to 512 rows.
//
// What bounds it.  As two kernels the weights and G are read twice, and dX's MFMA-bound pass stands in front of the update's
// HBM-bound one: 512 rows x 131,072 labels x 768 dims 330 us with the reduction, 1,310,720 labels 2.79 ms.  In one pass 235 and
// 2.24 ms.  Taken apart at 131,072 labels: the MFMAs with their LDS reads and the update take 172 us by themselves (82 of them the
// matrix pipes' at 2.4 GHz), weights, momentum and partial sums through HBM 170 (5.0 TB/s), and G adds 35 from HBM and 10 to 15 out
// of the L2, which every slice of dims reads it from: with slices of 64 dims, half as many registers for the sums, that was
// twice as much, and the pass took 300.
//
// Split.  A workgroup, one per CU, owns 128 dims and every a.ranges-th tile of 64 labels.  Four waves, one per SIMD, with all 512
// registers: the sums of dX, 16 RB rows x 128 dims of each wave, take the accumulation registers (256 for 512 rows), X^T of the wave's 32
// dims and all rows half of the others.  So a wave makes dW of its dims for all labels, 32 at a time, with G's fragments the only
// operand read from the LDS, and dX of its rows for all dims.  G lies in the LDS as two images of a tile, weights and momentum as two
// halves of one; everything travels by global->LDS fetches, so that nothing in flight holds a register.
//
// Schedule.  Half a tile is 16 RB MFMAs of a wave, dW's and then dX's; each is followed by its share of the rest: fragments of G
// twelve MFMAs ahead, every third one a fetch, the update of the half's 32 labels under dX's.  One barrier a half, before the
// last 18 MFMAs; the fetches of the next half's weights and momentum and of the next tile's G follow it, and the next half's first
// fragments.  A wave waits for the fetches by count: vector-memory operations retire in order.  The order itself is back_wide_order.hpp's.
// Stores of 16 labels x 64 bytes, half lines that the neighbouring wave completes, cost nothing against whole lines here.
//
// Layouts.  G's image: rows of 64 labels, read along the labels (dX) and transposed (dW).  The 16-byte chunk c of row r lies at
// c ^ g_swz(r): bits 1 and 2 of the XOR differ among the rows {0..3, 8..11} that half a wave's transposing read touches two by two
// to a bank line, all three among the eight even or odd rows of a straight one.  Weights and momentum: rows of 128 dims, swizzle of
// wide_core.hpp.  MFMA operands as in small_step.hpp, i = lane % 16, g = lane / 16.
//
// MFMAs, fetches and stores are inline asm, so the compiler keeps no distance between them and its own instructions: results are read
// ten slots after the last MFMA or more, bases of fetches and stores that may have been spilled go through a scalar move.
#pragma once
#include "back_step.hpp"
#include "back_wide_order.hpp"
#include "wide_core.hpp"

namespace xfc {

constexpr int BACK_WIDE_ROWS = 512;

// Up to 64 RB rows.
template <int RB_>
struct BackWide : BackWideOrder<RB_> {
  static constexpr int RB = RB_, NT = 256, ROWS = 64 * RB;
  static constexpr int G_BYTES = ROWS * BACK_TILE * 2, W_BYTES = BACK_DIMS * BACK_TILE;  // an image of G; of half a tile's weights
  static constexpr int LDS_BYTES = 2 * G_BYTES + 4 * W_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024 && ROWS <= BACK_WIDE_ROWS, "budget");

  // XOR on the 16-byte chunks of a row of G's image (128 bytes), and of the weights' (256)
  static __device__ __forceinline__ int g_swz(int row) {
    const int h = row >> 1;
    return (h & 4) | ((h & 1) << 1) | ((h >> 1) & 1);
  }
  static __device__ __forceinline__ int w_swz(int row) { return wide_mc_swz(row); }
  static __device__ __forceinline__ void tr(uint32_t at, half8& f, int half) {  // half of a transposing read
    const fp16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4f16((XFC_LDS fp16x4_t*)(uintptr_t)at);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * half + e] = (half_t)v[e];
  }
  static __device__ __forceinline__ half8 read16(uint32_t at) { return *(XFC_LDS const half8*)(uintptr_t)at; }
  static __device__ __forceinline__ void write16(uint32_t at, const half8& v) { *(XFC_LDS half8*)(uintptr_t)at = v; }
};

// f(integral_constant) for 0 .. N - 1: the schedule is compile-time arithmetic on a slot's number
template <int... I, class F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void each(F&& f) { each_of(std::make_integer_sequence<int, N>{}, f); }

// address = uniform 64-bit base + per-lane 32-bit offset (a store's data may not be overwritten by the next two instructions)
template <class V>
__device__ __forceinline__ void wide_store16(int64_t ubase, uint32_t voff, const V& v) {
  const uint64_t b = (uint64_t)uniform64(ubase);
  uint64_t t;  // see wide_load16
  asm volatile("s_mov_b64 %0, %3\n\tglobal_store_dwordx4 %1, %2, %0\n\ts_nop 1" : "=&s"(t) : "v"(voff), "v"(v), "s"(b) : "memory");
}
__device__ __forceinline__ void lane_load16(const void* p, uint32_t lds, int at) {
  const uint32_t m = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds);
  asm volatile("s_add_u32 m0, %0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m), "v"(p), "n"(at) : "memory", "m0", "scc");
}

#define XFC_INLINE __attribute__((always_inline))

// NT: weights and momentum are loaded as what will not be wanted again, for sizes that no cache holds until the next step.
template <class S, bool NT>
__global__ void __launch_bounds__(S::NT, 1) back_wide_kernel(BackArgs a) {
  constexpr int RB = S::RB, RP = S::RP, DW = S::DW, N = S::N;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const uint32_t gs = lds_addr(smem_raw);        // [2 images][ROWS][64 labels]
  const uint32_t ws = gs + 2 * S::G_BYTES;       // [2 halves][32 labels][128 dims]
  const uint32_t ms = ws + 2 * S::W_BYTES;       // the same
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int per = (int)gridDim.x >> 3, id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (id >= a.slices * a.ranges) return;
  const int slice = id % a.slices, range = id / a.slices, dim0 = slice * BACK_DIMS;
  const int part0 = range * a.parts, part1 = part0 + a.parts;
  // Its tiles: every a.ranges-th from the range's number on, counted from 0 here (a.back: from the last one on).
  const int t1 = (a.tiles - range + a.ranges - 1) / a.ranges, most = (a.tiles + a.ranges - 1) / a.ranges;
  const int whole = a.L - (a.tiles - 1) * BACK_TILE;                                     // labels of the last tile
  const int edge = whole < BACK_TILE && (a.tiles - 1) % a.ranges == range ? (a.back ? 0 : t1 - 1) : -1;  // if it is not whole and here
  const int label0 = (range + (a.back ? (t1 - 1) * a.ranges : 0)) * BACK_TILE, step = (a.back ? -a.ranges : a.ranges) * BACK_TILE;
  // Rows of the batch in an image: in their order, but for the last wave's, which are the batch's last 16 RB rounded up to eights;
  // those of them that another wave has, and those past the batch, are zeros.
  const int eights = (a.B + 7) >> 3, q0 = wave < 3 ? S::G_FETCH * wave : eights - S::G_FETCH;  // the wave's first eight
  const bool ragged = wave == 3 && a.B < S::ROWS;
  auto has = [&](int row) XFC_INLINE { return row >= 16 * RB * wave && row < a.B; };

  // What a lane fetches: row lane / 8 of an instruction's eight of G, 16 of its 128 bytes; row lane / 16 of four of weights.
  auto g_col = [&](int eight, int lane) XFC_INLINE { return 8 * ((lane & 7) ^ S::g_swz(8 * eight + (lane >> 3))); };
  const uint32_t lds_g = gs + (uint32_t)wave * (uint32_t)(S::G_FETCH * 1024);
  uint32_t gv[3];  // of even and odd eights; gv[2]: of the last, which may be part of one
  auto whole_g = [&]() XFC_INLINE {
    int lane_ = lane;
    asm volatile("" : "+v"(lane_));  // opaque: made once or twice, nothing of it is to be kept
#pragma unroll
    for (int h = 0; h < 2; ++h) gv[h] = (uint32_t)(lane_ >> 3) * (uint32_t)(a.ldg * 2) + 2u * g_col(h, lane_);
    const int last = a.B - 1 - 8 * (q0 + S::G_FETCH - 1);
    gv[2] = (uint32_t)((lane_ >> 3) < last ? lane_ >> 3 : last) * (uint32_t)(a.ldg * 2) + 2u * g_col(1, lane_);
  };
  whole_g();
  const uint32_t w_col = 16u * (uint32_t)((lane & 15) ^ S::w_swz(8 * wave + (lane >> 4)));
  const uint32_t wv = (uint32_t)(lane >> 4) * (uint32_t)(a.ldw * 2) + w_col;
  const int64_t w_row = uniform64(a.ldw * 2), w_step = uniform64((int64_t)step * a.ldw * 2);
  const int64_t g_step = (int64_t)step * 2, g_eight = uniform64(a.ldg * 16);
  int64_t at_g = uniform64(reinterpret_cast<int64_t>(a.G + (int64_t)(8 * q0) * a.ldg + label0));
  int64_t at_w = uniform64(reinterpret_cast<int64_t>(a.W + (int64_t)label0 * a.ldw + dim0));  // of the tile being multiplied
  const int64_t w_to_m = uniform64(reinterpret_cast<int64_t>(a.Mo) - reinterpret_cast<int64_t>(a.W));
  // To be called before the fetches of G of the tile that is not whole: labels past the end repeat others that are there.
  auto edge_g = [&]() XFC_INLINE {
#pragma unroll
    for (int h = 0; h < 3; ++h) {
      const int c = g_col(h > 0, lane);
      gv[h] -= c < whole ? 0u : 2u * c;
    }
  };
  // Zeros for what has come in place of rows and labels that are none: by the wave that fetched it, before the barrier.
  auto clear_g = [&](int tile, uint32_t image) XFC_INLINE {
    const int labels = tile == edge ? whole : BACK_TILE;
    int lane_ = lane;
    asm volatile("" : "+v"(lane_));  // opaque: rarely run, nothing of it is to be kept through the loop
#pragma unroll
    for (int j = 0; j < S::G_FETCH; ++j)
      if (!has(8 * (q0 + j) + (lane_ >> 3)) || g_col(j, lane_) >= labels) S::write16(image + j * 1024 + lane_ * 16, half8{});
  };
  auto clear_w = [&](int half) XFC_INLINE {
    int lane_ = lane;
    asm volatile("" : "+v"(lane_));
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (32 * half + 8 * wave + 4 * e + (lane_ >> 4) >= whole) S::write16(ws + half * S::W_BYTES + wave * 2048 + e * 1024 + lane_ * 16, half8{});
  };
  // The tiles come one after the other; `more`: the tile after this one is the range's too (else it is fetched again, so that
  // every tile has as many fetches as the counts of the waits assume).
  auto fetch_g = [&](auto j_, uint32_t image, bool more) XFC_INLINE {
    constexpr int j = decltype(j_)::value;
    wide_load16(at_g, gv[j == S::G_FETCH - 1 ? 2 : j & 1], image, j * 1024);
    at_g += j < S::G_FETCH - 1 ? g_eight : (more ? g_step : 0) - (S::G_FETCH - 1) * g_eight;
  };
  // weights (f = 0, 1) or momentum (2, 3) of half a tile, the one after `tile` if `next`
  auto fetch_w = [&](auto f_, auto half_, int tile, bool next) XFC_INLINE {
    constexpr int f = decltype(f_)::value, half = decltype(half_)::value, e = f & 1;
    next = next && tile + 1 < t1;
    const int first = 32 * half + 8 * wave + 4 * e;
    uint32_t v = wv;
    int64_t at = at_w + (f >= 2 ? w_to_m : 0) + (next ? w_step : 0) + first * w_row;
    if (tile + (next ? 1 : 0) == edge) {
      const int left = whole - 1 - first;  // the last label there is, from the instruction's first
      int lane_ = lane;
      asm volatile("" : "+v"(lane_));
      at += left < 0 ? left * w_row : 0;
      v = (uint32_t)((lane_ >> 4) < left ? lane_ >> 4 : left > 0 ? left : 0) * (uint32_t)(a.ldw * 2) + w_col;
    }
    wide_load16<NT, true>(at, v, (f < 2 ? ws : ms) + half * S::W_BYTES + wave * 2048, e * 1024);
  };

  // X^T, A side of dW: rows 8 g ..+7 of each 32, dim 8 (i / 4) + 4 b + i % 4 of the wave's 32.  By way of G's images, 64 dims each.
  const int k0 = 8 * g + (i >> 2);  // row of a transposing read's first half (mod 32), the second's is four on
  half8 xt[RP][2];
  each<2 * S::G_FETCH>([&](auto j_) XFC_INLINE {
    constexpr int j = decltype(j_)::value % S::G_FETCH, image = decltype(j_)::value / S::G_FETCH;
    const int row = 8 * (q0 + j) + (lane >> 3);
    lane_load16(has(row) ? (const void*)(a.X + (int64_t)row * a.ldx + dim0 + 64 * image + g_col(j, lane)) : (const void*)g_zero16,
                lds_g + image * S::G_BYTES, j * 1024);
  });
  wait_vmcnt_barrier<0>();
#pragma unroll
  for (int p = 0; p < RP; ++p)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint32_t at = gs + (wave >> 1) * S::G_BYTES + k0 * 128 + 16 * ((4 * (wave & 1) + (i & 3)) ^ S::g_swz(k0)) + 8 * b + 4096 * p;
      S::tr(at, xt[p][b], 0);
      S::tr((at ^ 16) + 512, xt[p][b], 1);
    }
  Wave16::barrier();
  if (edge == 0) edge_g();
  each<S::G_FETCH>([&](auto j) XFC_INLINE { fetch_g(j, lds_g, 1 < t1); });
  each<4>([&](auto f) XFC_INLINE {
    fetch_w(f, std::integral_constant<int, 0>{}, 0, false);
    fetch_w(f, std::integral_constant<int, 1>{}, 0, false);
  });
  if (edge == 0 && t1 > 1) whole_g();
  if (edge == 1) edge_g();
  wait_vmcnt<0>();
  if (ragged || edge == 0) clear_g(0, lds_g);
  if (edge == 0) clear_w(0);
  Wave16::barrier();

  // LDS addresses of a lane's reads.  In G's images rows four apart have their chunks XORed by 1 more.
  const uint32_t b0 = 8u * (i & 1), c0 = (i & 3) >> 1;
  const uint32_t gt_at = gs + k0 * 128 + (c0 ^ S::g_swz(k0)) * 16 + b0;                        // transposing: rows k0.., labels 4 (i % 4) ..+3
  const uint32_t wt_at = ws + k0 * 256 + (c0 ^ S::w_swz(k0)) * 16 + b0;                        // transposing: labels k0.., dims 4 (i % 4) ..+3
  const uint32_t bg_at = gs + (16 * RB * wave + i) * 128 + (g ^ S::g_swz(i)) * 16;             // row 16 RB wave + i, labels 8 g ..+7
  const uint32_t own_at = ws + i * 256 + ((4 * wave + g) ^ S::w_swz(i)) * 16;                  // label i, dims 32 wave + 8 g ..+7
  const uint32_t w_out = (uint32_t)i * (uint32_t)(a.ldw * 2) + 64u * wave + 16u * g;

  float4v acc[RB][8];  // rows 16 (RB wave + rb) + i, dims 16 c + 4 g ..+3
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      acc[rb][c] = float4v{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[rb][c]));
    }
  // The sums of a part leave when the tile before `upto` ends it (they may be none, as may the tiles of a part).
  auto first_tile = [&](int part) XFC_INLINE { return part < part1 ? (int)((int64_t)most * (part - part0) / a.parts) : t1; };
  int part = part0, end = first_tile(part0 + 1);
  auto leave = [&](int upto) XFC_INLINE {
    if (part >= part1 || end != upto) return;
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
    do {
      int lane_ = lane;
      asm volatile("" : "+v"(lane_));
      int row = 8 * q0 + (lane_ & 15);
      const int at = dim0 + 4 * (lane_ >> 4);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        float* dst = a.part + ((int64_t)part * a.B + row) * a.d + at;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          float4v v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float x;
            asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(acc[rb][c][e]));
            v[e] = x;
          }
          if (has(row)) *reinterpret_cast<float4v*>(dst + 16 * c) = v;
          acc[rb][c] = float4v{0.f, 0.f, 0.f, 0.f};
          asm volatile("" : "+a"(acc[rb][c]));
        }
        row += 16;
        __builtin_amdgcn_sched_barrier(0);
      }
      end = first_tile(++part + 1);
    } while (part < part1 && end == upto);
    asm volatile("s_nop 7" ::: "memory");  // cleared registers on their way into MFMAs
  };
  leave(0);

  uint32_t g_off = 0;  // image of the tile being multiplied
  half8 gt[RP][2];     // [rows 32 p ..+31][labels 16 lb ..+15]; the first ones are read at the end of the half before
  each<4 * S::AHEAD>([&](auto r_) XFC_INLINE {
    constexpr int r = decltype(r_)::value, lb = (r >> 1) & 1;
    S::tr(((gt_at ^ 32 * lb) ^ 16 * (r & 1)) + 512 * (r & 1) + 4096 * (r >> 2), gt[r >> 2][lb], r & 1);
  });
  each<S::TAIL - 4>([&](auto j) XFC_INLINE { fetch_g(j, lds_g + S::G_BYTES, 2 < t1); });

  for (int tile = 0; tile < t1; ++tile) {
    auto half = [&](auto half_) XFC_INLINE {
      constexpr int h = decltype(half_)::value;
      const uint32_t gt0 = (gt_at + g_off) ^ 64 * h, bg0 = (bg_at + g_off) ^ 64 * h;
      const uint32_t gt1 = h ? gt_at + (S::G_BYTES - g_off) : (gt_at + g_off) ^ 64;  // of the next half
      const uint32_t lds_here = lds_g + g_off, lds_next = lds_g + (S::G_BYTES - g_off);
      half8 bg[RB], wt[8], wq[2], mq[2];
      float4v dw[2][2];  // [labels 16 lb + i][dims 32 wave + 8 g + 4 b ..+3]
      float gg[2], mf[2];
      auto update = [&](auto piece) XFC_INLINE {  // of two elements, a step of the arithmetic
        constexpr int u = decltype(piece)::value, v = u < 16 ? u : u - 17, lb = u < 16 ? 0 : 1, e0 = 2 * ((v >> 2) & 3);
        if constexpr (v >= 0 && v < 16) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            if constexpr (v % 4 == 0) gg[q] = dw[lb][e0 >> 2][(e0 & 3) + q] + a.wd * (float)wq[lb][e0 + q];
            if constexpr (v % 4 == 1) mf[q] = a.mu * (float)mq[lb][e0 + q] + gg[q];
            if constexpr (v % 4 == 2) mq[lb][e0 + q] = (half_t)mf[q];
            if constexpr (v % 4 == 3) wq[lb][e0 + q] = (half_t)((float)wq[lb][e0 + q] - a.lr * mf[q]);
          }
        }
      };
      auto store = [&](auto lb_) XFC_INLINE {
        constexpr int lb = decltype(lb_)::value;
        const int64_t to = at_w + (32 * h + 16 * lb) * w_row;
        auto out = [&]() XFC_INLINE {
          wide_store16(to + w_to_m, w_out, mq[lb]);
          wide_store16(to, w_out, wq[lb]);
        };
        if (tile != edge) {
          out();
        } else {
          int lane_ = lane;
          asm volatile("" : "+v"(lane_));
          if (32 * h + 16 * lb + (lane_ & 15) < whole) out();
        }
      };
      each<N>([&](auto slot) XFC_INLINE {
        constexpr int n = decltype(slot)::value;
        if constexpr (n == S::BAR) {
          if (tile == edge) wait_vmcnt<S::wait(h, true)>();
          if constexpr (h == 0) {
            if (tile == edge) clear_w(1);
          } else if (ragged || tile + 1 == edge) {
            wait_vmcnt<S::wait(h, false)>();
            clear_g(tile + 1, lds_next);
            if (tile + 1 == edge) clear_w(0);
          }
          wait_lds_vmcnt_barrier<S::wait(h, false)>();
          if constexpr (h == 1) {
            if (tile + 2 == edge) edge_g();
          }
        }
        if constexpr (n < DW) {
          constexpr int p = n >> 2, lb = (n >> 1) & 1, b = (n ^ lb) & 1;
          if constexpr (p == 0) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=&v"(dw[lb][b]) : "v"(xt[p][b]), "v"(gt[p][lb]));
          else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(dw[lb][b]) : "v"(xt[p][b]), "v"(gt[p][lb]));
        } else {
          constexpr int rb = (n - DW) >> 3, c = (n - DW) & 7;
          asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[rb][c]) : "v"(wt[c]), "v"(bg[rb]));
        }
        // fragments
        if constexpr (n < 4 * (RP - S::AHEAD)) {
          constexpr int lb = (n >> 1) & 1;
          S::tr(((gt0 ^ 32 * lb) ^ 16 * (n & 1)) + 512 * (n & 1) + 4096 * ((n >> 2) + S::AHEAD), gt[(n >> 2) + S::AHEAD][lb], n & 1);
        }
        constexpr int w = n - (DW > 34 ? DW - 34 : 0);
        if constexpr (w >= 0 && w < 32 && w % 2 == 0) S::tr((wt_at ^ 32 * (w >> 2)) + h * S::W_BYTES + 1024 * ((w >> 1) & 1), wt[w >> 2], (w >> 1) & 1);
        constexpr int q = n - (DW - 9);
        if constexpr (q >= 0 && (q < 8 ? q % 4 == 0 : q % 8 == 4)) {
          constexpr int rb = q < 8 ? q / 4 : q / 8 + 1;
          if constexpr (rb < RB) bg[rb] = S::read16(bg0 + 2048 * rb);
        }
        constexpr int r = n - S::BAR - 1;
        if constexpr (r >= 0 && r < 4 * S::AHEAD) {
          constexpr int lb = (r >> 1) & 1;
          S::tr(((gt1 ^ 32 * lb) ^ 16 * (r & 1)) + 512 * (r & 1) + 4096 * (r >> 2), gt[r >> 2][lb], r & 1);
        }
        if constexpr (n == S::UPD - 6) wq[0] = S::read16(own_at + h * S::W_BYTES);
        if constexpr (n == S::UPD - 4) mq[0] = S::read16(own_at + (2 + h) * S::W_BYTES);
        if constexpr (n == S::STORE0 - 6) wq[1] = S::read16(own_at + h * S::W_BYTES + 4096);
        if constexpr (n == S::STORE0 - 4) mq[1] = S::read16(own_at + (2 + h) * S::W_BYTES + 4096);
        // fetches
        if constexpr (constexpr int f = S::w_fetch(n); f >= 0) fetch_w(std::integral_constant<int, f>{}, std::integral_constant<int, h>{}, tile, true);
        if constexpr (constexpr int j = S::g_fetch(h, n); j >= 0) {
          if constexpr (h == 1) fetch_g(std::integral_constant<int, j>{}, lds_here, tile + 3 < t1);
          else fetch_g(std::integral_constant<int, j>{}, lds_next, tile + 2 < t1);
        }
        if constexpr (n >= S::UPD && n <= S::STORE1)
          each<S::PACE>([&](auto u) XFC_INLINE { update(std::integral_constant<int, S::PACE * (n - S::UPD) + decltype(u)::value>{}); });
        if constexpr (n == S::STORE0) store(std::integral_constant<int, 0>{});
        if constexpr (n == S::STORE1) store(std::integral_constant<int, 1>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
    at_w += w_step;
    g_off = S::G_BYTES - g_off;
    leave(tile + 1);
  }
  wait_vmcnt<0>();
}

}  // namespace xfc
