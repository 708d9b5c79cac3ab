// Both products of the backward pass in one pass over the labels, for batches of up to 256 rows: dX += G.W from the weights
// before the update, and dW = G^T.X, which is written out or consumed by the momentum update of those weights.
//
// What bounds it.  With so few rows the products are small beside the traffic; as two kernels the weights and G were read
// twice.  dX and the update of 199 rows x 131,072 labels x 768 dims, reduction included: 239 -> 199 us (256 rows 248 -> 220, 128
// rows 202 -> 183: 5.0 TB/s of the 8 bytes per weight and G); without its stores the pass took 150 at 199 and 256 rows, the LDS
// reads and their latency between two barriers.  Above 192 rows the sums of one tile that dX is made from (one rounding each into
// the running sum) take the registers of half of X^T: 211 -> 220 us at 256 rows, dX as close to float64 as xfc_dx's.  Whole steps of 65 to 256 rows x 4,001 to 2,812,281 labels x 64 to 1024 dims: 1.03
// to 1.5 times as fast.
//
// Split.  A workgroup owns a slice of 128 dims and every a.ranges-th tile of 64 labels, from the last one on.  Its eight waves are two
// groups of 64 dims by four quarters; a quarter takes 16 of the tile's labels for dW and their update, and a quarter of the
// rows for dX.  The weights cross between the quarters, and G between all, through the LDS, with one barrier a tile (two
// images of each); X^T stays in the registers as far as they reach, the rest lies in the LDS as MFMA fragments, and dX stays in
// the registers.  The weights and the momentum of the next two tiles are on their way, fetched unconditionally (past the last
// tile it again), so that the waits count the loads exactly; G goes straight to the LDS, a tile ahead.  The slices of a range
// run side by side on one XCD and meet in its L2 for G.
//
// Order.  The whole chip walks from the last labels to the first, as the forward pass has left the caches the last ones' G and weights
// (up to 256 MB of them), and ends with those that the next forward pass begins with.  Each range a stretch of its own, from its first
// label on -> this, whole steps: 256 rows x 131,072 labels x 768 dims 272 -> 263 us, 100 x 400,001 x 384 331 -> 322, 90 x 2,000,000 x
// 128 639 -> 585, two micro-batches of 200 x 200,001 x 384 626 -> 596.  The fetches of G are dealt to the waves one by one, so that
// with 193 to 255 rows, or 129 to 191, all have some: 199 x 131,072 x 768 with the loss 291 -> 283, and with the non-temporal stores, which
// until then did not pay there, 261; 200 x 200,001 x 512 297 -> 267.  The first ones are sent before X^T is turned.
//
// Whole lines.  An instruction that loads or stores weights or momentum covers 8 labels x 128 bytes: lanes with i < 8 have
// dims 8 g ..+7 of label i, the others dims 32 + 8 g ..+7 of label i - 8.  The products come out 16 labels x 32 dims at a
// time, so half of them move eight lanes over before the update.  (16 labels x 64 bytes, the other halves of the lines by another
// wave: 258 us at 199 x 131,073 x 768; whole lines make it 222, non-temporal loads of them 213, G through the LDS alone and half
// of X^T in registers 202.)
//
// Register layouts: those of small_step.hpp, i = lane % 16, g = lane / 16.
#pragma once
#include "wave16.hpp"

namespace xfc {

constexpr int BACK_MAX_ROWS = 256, BACK_TILE = 64, BACK_AHEAD = 2;
enum BackMode { BACK_UPDATE = 0, BACK_OUT = 1, BACK_ADD = 2 };  // ADD: out = G^T.X + beta * out, else without the addend

struct BackArgs {
  const half_t* G; int64_t ldg;
  const half_t* X; int64_t ldx;
  half_t* W; int64_t ldw;                     // read only but for BACK_UPDATE
  half_t* Mo; int64_t ldm; float lr, mu, wd;  // BACK_UPDATE
  float* out; int64_t ldo; float beta;        // BACK_OUT, BACK_ADD
  float* part;                                // [ranges * parts][B][d] partial sums of G.W
  int B, L, d;
  int slices, ranges, parts, tiles;           // ranges a multiple of 8 (back_wide.hpp: any number); tiles of 64 labels
  bool back;                                  // back_wide.hpp: the last labels first
};

template <bool NT, class T>
__device__ __forceinline__ T load(const T* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// up to 64 RQ rows; XR of the 2 RQ blocks of 32 rows of X^T in registers
template <int RQ_, int XR_>
struct BackStep : Wave16 {
  static constexpr int RQ = RQ_, XR = XR_, NT = 512, ROWS = 64 * RQ, RP = 2 * RQ;
  static constexpr int G_HALVES = ROWS * BACK_TILE, W_HALVES = BACK_DIMS * BACK_TILE, X_HALVES = (RP - XR) * 32 * BACK_DIMS;
  static constexpr int LDS_BYTES = (X_HALVES + 2 * (G_HALVES + W_HALVES)) * 2;
  static constexpr int G_FETCH = ROWS / 64;  // fetch instructions (16 rows x 32 labels of G) of a wave per tile
  static_assert(LDS_BYTES <= 160 * 1024 && ROWS <= BACK_MAX_ROWS && XR <= RP, "budget");
};

// HOW the arrays that are written (BACK_UPDATE: W and Mo, otherwise out) are stored; PAST: and loaded, as what will not be wanted
// again.  THROUGH: the partial sums as well.
template <class S, int MODE, int HOW>
__global__ void __launch_bounds__(S::NT, 2) back_step_kernel(BackArgs a) {
  constexpr int RQ = S::RQ, RP = S::RP, XR = S::XR;
  constexpr bool NT = HOW == PAST;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* const gs = reinterpret_cast<half_t*>(smem_raw);  // [2 images][2 halves of the tile][ROWS][32]
  half_t* const ws = gs + 2 * S::G_HALVES;                 // [2 images][2 halves of the tile][4 blocks of 32 dims][32][32]
  half_t* const xs = ws + 2 * S::W_HALVES;                 // [RP - XR][2 groups][2 blocks][2][64 lanes][8]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int t4 = 8 * g + (i >> 2);  // row of a transposing read's first half
  const int dg = wave & 1, qt = wave >> 1;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int slice = local % a.slices, range = (local / a.slices) * 8 + xcd;
  const int dim0 = slice * BACK_DIMS + dg * 64;
  const int part0 = range * a.parts, part1 = part0 + a.parts;
  // Its tiles: every a.ranges-th from the range's number on, counted from the last one.
  const int t1 = (a.tiles - range + a.ranges - 1) / a.ranges, most = (a.tiles + a.ranges - 1) / a.ranges;
  auto l0_of = [&](int tile) { return (range + (t1 - 1 - tile) * a.ranges) * BACK_TILE; };
  auto first_tile = [&](int part) { return part < part1 ? (int)((int64_t)most * (part - part0) / a.parts) : t1; };
  const int low = i & 7, second = i >> 3;  // of the whole-line layout: label (and low + 8), which 32 dims (fp32: which 16)

  // What a thread fetches.  Labels, rows and dims past the end repeat the last ones; they are cleared in the LDS, or belong
  // to nothing that is stored.
  struct Ahead {
    half8 w[2], m[2];  // labels low and low + 8
    float4v o[2][2];   // BACK_ADD: [block of 32 dims][labels low, low + 8]
  } ahead[BACK_AHEAD];
  const int col = dim0 + 32 * second + 8 * g, colc = col < a.d ? col : a.d - 8;
  auto col32 = [&](int s) { return dim0 + 32 * s + 16 * second + 4 * g; };
  auto fetch = [&](int tile, Ahead& q) {
    const int l0 = l0_of(tile < t1 ? tile : t1 - 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int label = l0 + 16 * qt + 8 * h + low;
      const int64_t l = label < a.L ? label : a.L - 1;
      q.w[h] = load<NT && MODE == BACK_UPDATE>(reinterpret_cast<const half8*>(a.W + l * a.ldw + colc));
      if constexpr (MODE == BACK_UPDATE) q.m[h] = load<NT>(reinterpret_cast<const half8*>(a.Mo + l * a.ldm + colc));
      if constexpr (MODE == BACK_ADD) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int c = col32(s);
          q.o[s][h] = load<NT>(reinterpret_cast<const float4v*>(a.out + l * a.ldo + (c < a.d ? c : a.d - 4)));
        }
      }
    }
  };
  // A tile of G to an image: 16 rows x 32 labels an instruction, both halves of a line one after the other.  Rows past the
  // batch stay the zeros they were at the start, or come as such, and so do labels past the last eight.  The fetches are the
  // wave's last ones but for `after` loads and the tile's stores.
  auto fetch_g = [&](int tile, half_t* image) {
    const int l0 = l0_of(tile);
#pragma unroll
    for (int j = 0; j < S::G_FETCH; ++j) {
      const int n = 8 * j + wave, row0 = (n >> 1) * 16, k = n & 1, at = l0 + 32 * k;
      if (row0 < a.B) {
        half_t* const dst = image + (k * S::ROWS + row0) * 32;
        if (row0 + 16 <= a.B && at + 32 <= a.L) {
          load16_to_lds(a.G + (int64_t)row0 * a.ldg + at, (uint32_t)(lane >> 2) * (uint32_t)(a.ldg * 2) + 16u * (lane & 3), dst);
        } else {
          const int row = row0 + (lane >> 2), c = at + 8 * (lane & 3);
          load16_to_lds(row < a.B && c < a.L ? (const void*)(a.G + (int64_t)row * a.ldg + c) : (const void*)g_zero16, dst);
        }
      }
    }
  };
  if (t1 > 0) {
#pragma unroll
    for (int t = 0; t < BACK_AHEAD; ++t) fetch(t, ahead[t]);
    fetch_g(0, gs);
  }

  // X^T, A side of dW: rows 8 g ..+7 of each 32, dim 8 (i / 4) + 4 b + i % 4 of a block (in fp32: 16 b + i).  Rows past the
  // batch are zeros, as they are in the images of G.
  half8 xt[XR > 0 ? XR : 1][2][2];
  {
    half_t* const mine = ws + wave * 2048;
    auto turn = [&](int p, half8 (&x)[2][2]) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int rel = 8 * (i >> 2) + 4 * b + (i & 3), row = 32 * p + rel, c = dim0 + 32 * s + 8 * g;
          half8 v = {};
          if (row < a.B) v = *reinterpret_cast<const half8*>(a.X + (int64_t)row * a.ldx + (c < a.d ? c : a.d - 8));
          *reinterpret_cast<half8*>(mine + s * 1024 + rel * 32 + 8 * g) = v;
        }
      S::lds_done();
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          x[s][b] = S::read_tr(mine + s * 1024, t4, MODE == BACK_UPDATE ? 8 * (lane & 3) + 4 * b : 16 * b + 4 * (lane & 3));
      S::lds_done();
    };
#pragma unroll
    for (int p = 0; p < XR; ++p) turn(p, xt[p]);
    for (int p = XR + qt; p < RP; p += 4) {
      half8 x[2][2];
      turn(p, x);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b) *reinterpret_cast<half8*>(xs + ((((p - XR) * 2 + dg) * 2 + s) * 2 + b) * 512 + lane * 8) = x[s][b];
    }
    for (int q = tid; q < 4 * S::ROWS * 4; q += S::NT)
      if ((q >> 2) % S::ROWS >= a.B) *reinterpret_cast<half8*>(gs + q * 8) = half8{};
    S::barrier();  // X^T is whole, the images of the weights are free
  }
  float4v acc[RQ][4];  // rows 16 (RQ qt + rb) + i, dims 16 c + 4 g ..+3 of the group's 64
#pragma unroll
  for (int rb = 0; rb < RQ; ++rb)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[rb][c] = float4v{0.f, 0.f, 0.f, 0.f};
  // The sums of a part leave when the tile before `upto` ends it (they may be none, as may the tiles of a part).
  int part = part0, end = first_tile(part0 + 1);
  auto leave = [&](int upto) {
    while (part < part1 && end == upto) {
      int row = RQ * qt * 16 + i, at = dim0 + 4 * g;
      asm volatile("" : "+v"(row), "+v"(at));  // opaque: addresses made here and not kept through the loop
      float* dst = a.part + ((int64_t)part * a.B + row) * a.d + at;
#pragma unroll
      for (int rb = 0; rb < RQ; ++rb) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if (row < a.B && at + 16 * c < a.d) store<HOW == THROUGH ? THROUGH : CACHED>(reinterpret_cast<float4v*>(dst + 16 * c), acc[rb][c]);
          acc[rb][c] = float4v{0.f, 0.f, 0.f, 0.f};
        }
        row += 16;
        dst += 16 * (int64_t)a.d;
        __builtin_amdgcn_sched_barrier(0);
      }
      end = first_tile(++part + 1);
    }
  };
  leave(0);

  int parity = 0;
  // Loads and stores of a wave between its fetches of G and the barrier that makes them known: of tiles that are whole.
  constexpr int AFTER = MODE == BACK_UPDATE ? 8 : MODE == BACK_ADD ? 10 : 6;
  bool exact = false;
  auto work = [&](int tile, Ahead& q) {
    const int l0 = l0_of(tile), label = l0 + 16 * qt + low;
    half_t* const gi = gs + parity * S::G_HALVES;
    half_t* const wi = ws + parity * S::W_HALVES;
    parity ^= 1;
    Ahead now = q;
    if (l0 + BACK_TILE > a.L) {  // labels past the last one weigh nothing
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) now.w[h][e] = label + 8 * h < a.L ? now.w[h][e] : (half_t)0.f;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
      *reinterpret_cast<half8*>(wi + (((qt >> 1) * 2 + dg) * 2 + second) * 1024 + (16 * (qt & 1) + 8 * h + low) * 32 + 8 * g) = now.w[h];
    if (exact) wait_vmcnt<AFTER>();
    else wait_vmcnt<0>();
    S::barrier();
    if (tile + 1 < t1) fetch_g(tile + 1, gs + parity * S::G_HALVES);
    fetch(tile + BACK_AHEAD, q);
    exact = l0 + BACK_TILE <= a.L && dim0 + 64 <= a.d;  // every lane stores
    // dX^T += W^T . G^T, this quarter's rows: the tile's 64 labels by themselves, then one addition.  (An MFMA rounds its sum
    // once per 16 of k, and the error of a long sum grows with the root of its roundings: see back_plan.)
    {
      half8 bg[2][RQ];
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int rb = 0; rb < RQ; ++rb)
          bg[k][rb] = *reinterpret_cast<const half8*>(gi + (k * S::ROWS + (RQ * qt + rb) * 16 + i) * 32 + 8 * g);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float4v t[RQ];
#pragma unroll
        for (int rb = 0; rb < RQ; ++rb) t[rb] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const half8 wt = S::read_tr(wi + ((k * 2 + dg) * 2 + (c >> 1)) * 1024, t4, 16 * (c & 1) + 4 * (lane & 3));
#pragma unroll
          for (int rb = 0; rb < RQ; ++rb) t[rb] = S::mfma(wt, bg[k][rb], t[rb]);
        }
#pragma unroll
        for (int rb = 0; rb < RQ; ++rb) {
          acc[rb][c] += t[rb];
          asm volatile("" : "+v"(acc[rb][c]));  // added here: the sums of all blocks, kept for later, would not fit the registers
        }
      }
    }
    // dW^T = X^T . G, this quarter's labels
    float4v dw[2][2];  // label 16 qt + i; UPDATE: dims 8 g + 4 b ..+3 of block s, else 16 b + 4 g ..+3
#pragma unroll
    for (int s = 0; s < 2; ++s) dw[s][0] = dw[s][1] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const half8 gt = S::read_tr(gi + ((qt >> 1) * S::ROWS + 32 * p) * 32, t4, 16 * (qt & 1) + 4 * (lane & 3));
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          if (p < XR) dw[s][b] = S::mfma(xt[p < XR ? p : 0][s][b], gt, dw[s][b]);
          else dw[s][b] = S::mfma(*reinterpret_cast<const half8*>(xs + ((((p - XR) * 2 + dg) * 2 + s) * 2 + b) * 512 + lane * 8), gt, dw[s][b]);
        }
    }
    if constexpr (MODE == BACK_UPDATE) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        half8 wv = now.w[h], mv = now.m[h];
        float4v d4[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const float4v far = S::across8(dw[1 - h][b]);
#pragma unroll
          for (int e = 0; e < 4; ++e) d4[b][e] = second == h ? dw[h][b][e] : far[e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float wf = (float)wv[e];
          const float gg = d4[e >> 2][e & 3] + a.wd * wf;
          const float mf = a.mu * (float)mv[e] + gg;
          mv[e] = (half_t)mf;
          wv[e] = (half_t)(wf - a.lr * mf);
        }
        if (label + 8 * h < a.L && col < a.d) {
          store<HOW>(reinterpret_cast<half8*>(a.Mo + (int64_t)(label + 8 * h) * a.ldm + col), mv);
          store<HOW>(reinterpret_cast<half8*>(a.W + (int64_t)(label + 8 * h) * a.ldw + col), wv);
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float4v far = S::across8(dw[s][1 - h]);
          float4v v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = second == h ? dw[s][h][e] : far[e];
          if constexpr (MODE == BACK_ADD) v += a.beta * now.o[s][h];
          if (label + 8 * h < a.L && col32(s) < a.d)
            store<HOW>(reinterpret_cast<float4v*>(a.out + (int64_t)(label + 8 * h) * a.ldo + col32(s)), v);
        }
    }
    leave(tile + 1);
  };
  for (int t = 0; t < t1; t += BACK_AHEAD) {
#pragma unroll
    for (int s = 0; s < BACK_AHEAD; ++s)
      if (t + s < t1) work(t + s, ahead[s]);  // (the barriers: every wave has the same tiles)
  }
}

}  // namespace xfc
