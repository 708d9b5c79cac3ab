// The whole step of a batch of up to 64 rows in one pass over the labels: every weight and every momentum is read once
// and written once, which is all that such a step has to move.
//
// What bounds it.  The step's products are small (16 to 64 rows against each weight), its traffic is not: 8 bytes per
// weight.  As three products the weights came from memory twice more, and each launch filled and drained the chip anew.
// Whole steps, three passes -> one: 32 rows x 131,072 labels x 768 dims 245 -> 193 us and with whole lines (LINES below) 171
// (this kernel 166: 4.9 TB/s of those 8 bytes); 8 x 40,001 x 128 96 -> 23 us; 64 x 400,001 x 384 471 -> 307 us.  What is left:
// where whole lines do not pay, the weights' and the momentum's loads come in pieces of 64 bytes, and a small label count is
// one tile to a workgroup, a chain of loads, z, the two barriers and the update (17 to 27 us).
//
// Split.  A workgroup takes tiles of 32 labels; each of its NW waves owns D / NW of the dims of all of them, for all three
// products, so that a weight is loaded by one lane, used from its registers for z and for the update, and stored by the
// same lane.  What crosses waves is z alone (each wave has the part of its dims): summed through the LDS in wave order.
// While a tile is worked on, the next tile's weights and this tile's momentum are on their way.
//
// Register layouts (MFMA 16x16x32, see wide_core.hpp).  i = lane % 16, g = lane / 16:
//   W        lane holds W[label 16 lb + i][32 s + 8 g ..+7]: as it lies in memory, and the B side of z = X.W^T
//   z        the A side's rows are those of X permuted inside every 32 (row 8 (i / 4) + 4 b + i % 4 for block b), so that
//            a lane's registers are rows 8 g + 4 b ..+3 of label 16 lb + i
//   G        goes through the LDS as [row][label]: read as rows it is the B side of dX^T = W^T.G^T and what is stored,
//            read transposed the B side of dW^T = X^T.G^T
//   dW       the A side's dims are permuted like the rows above, so the two blocks of 32 dims give a lane dims
//            8 g ..+7 of label 16 lb + i: those of the weights it holds
//   dX       lane holds dims 4 g ..+3 of row 16 rb + i, accumulated over all tiles of the workgroup
#pragma once
#include "wave16.hpp"

namespace xfc {

// More rows than 64 do not fit the registers; label pairs are held 3 to 8 to a thread.
constexpr int SMALL_MAX_ROWS = 64, SMALL_MAX_PAIRS = 2048;

struct SmallArgs {
  const half_t* X; int64_t ldx;
  half_t* W; int64_t ldw;
  half_t* Mo; int64_t ldm;
  half_t* G; int64_t ldg;
  const int32_t* rowptr; const int32_t* colidx;  // CSR, or
  const int64_t* pos_x; const int64_t* pos_y;    // COO if pos_x is given
  int nnz, B, L, n_store, tiles;                 // n_store = L rounded up to 8: those columns of G are written as zero
  float lr, mu, wd;
  float* part;                                   // [gridDim.x][B][D] partial sums of G.W
};

// NW waves, SB blocks of 32 dims per wave, RB blocks of 16 rows (2 or 4); LINES: an instruction that loads or stores weights
// or momentum covers 8 labels x 128 bytes (see back_step.hpp) instead of 16 x 64, and the loads and stores say that nothing will
// want them again.  That is for sizes that no cache holds until the next step: 32 rows x 131,072 x 768 188 -> 169 us, x 700,001 961 ->
// 888, 64 x 700,001 x 512 696 -> 621 (whole lines without the hint 720, half lines with it 1,048 at 32 x 700,001 x 768).  The stores' hint
// alone, 32 x 131,072 x 768: back to back 171 -> 158, each step followed by a copy of 512 MiB 374 -> 361 or by 0.6 ms of matrix products
// 767 -> 763, a new state's first 182 -> 179, waited for 165 -> 183, when whoever runs next need not write back what the caches hold.  Below,
// half lines without the hint are faster, as the caches serve them: 64 x 20,011 x 512 33.0 against 34.5, 32 x 4,097 x 1024 24.8
// against 28.1.
template <int NW_, int SB_, int RB_, bool LINES_ = false>
struct SmallStep : Wave16 {
  static constexpr int NW = NW_, SB = SB_, RB = RB_, P = RB / 2, NT = 64 * NW, D = NW * SB * 32;
  static constexpr int UNITS = 2 * RB;           // 16 x 16 blocks of z, each summed by one wave
  static constexpr bool SKIP = UNITS == NW;      // one block per wave: its own part need not go through the LDS
  static constexpr int SLOTS = SKIP ? UNITS - 1 : UNITS;
  static constexpr int X_BYTES = 16 * RB * D * 2;
  static constexpr int REGION = SLOTS * 1024 > SB * 2048 ? SLOTS * 1024 : SB * 2048;  // per wave: parts of z, then its W
  static constexpr int G_BYTES = 16 * RB * 64, MASK_WORDS = P * 32;
  static constexpr int LDS_BYTES = X_BYTES + NW * REGION + G_BYTES + 2 * MASK_WORDS * 4;
  static constexpr int PAIRS = (SMALL_MAX_PAIRS + NT - 1) / NT;  // label pairs a thread holds
  // Workgroups per CU: as many as the registers (256 a wave, 128 with one block of dims and 32 rows, 168 with 12 waves) and the LDS allow.
  static constexpr int WAVES_PER_EU = NW == 12 ? 3 : SB == 1 && RB == 2 ? 4 : 2;
  // With 32 rows the next tile's weights and momentum are both fetched while a tile is worked on.  With more rows, or 128
  // dims a wave, the registers do not hold them beside the sums (40 to 60 spilled, 749 us instead of 618 at 64 rows x
  // 400,001 labels x 768): there the momentum's loads wait until z has left its registers, and the weights move to the LDS
  // after that and the next tile's are fetched in their place.  Spills that are left: 22 registers at 64 rows x 768, 5 at
  // 32 x 128, 2 at 32 x 384.
  static constexpr bool AHEAD = RB == 2 && SB <= 3;
  static constexpr bool LINES = LINES_;
  static_assert(!LINES || SB % 2 == 0, "a line is two blocks of dims");
  static constexpr int BY_REGS = 4 * WAVES_PER_EU / NW, BY_LDS = 160 * 1024 / LDS_BYTES;
  static constexpr int PER_CU = BY_REGS < BY_LDS ? BY_REGS : BY_LDS;
  static_assert(LDS_BYTES <= 160 * 1024 && PER_CU >= 1, "LDS and register budget");
  static_assert(UNITS % NW == 0 || UNITS < NW, "blocks of z divide among the waves");
  static_assert(RB <= NW, "one wave stores 16 rows of G");
};

// 1 / (1 + 2^(-z log2 e)) with the bare v_exp_f32 / v_rcp_f32: the exponential may flush to zero or
// overflow to infinity at the ends, where the quotient is 1 or 0 either way, so the range fix-up that
// __expf carries (a compare and a select per element) buys nothing here.
__device__ __forceinline__ float sigmoidf_fast(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.44269504088896341f));
}

// STEP false: G alone, the first half of the step (W is only read; Mo and part are not used).
template <class S, bool STEP = true>
__global__ void __launch_bounds__(S::NT, S::WAVES_PER_EU) small_step_kernel(SmallArgs a) {
  constexpr bool AHEAD = S::AHEAD || !STEP;  // without the momentum and the sums the next tile's weights always fit
  constexpr int NW = S::NW, SB = S::SB, RB = S::RB, P = S::P, D = S::D;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int t4 = 8 * g + (i >> 2);   // row of a transposing read's first half
  const int dim0 = wave * SB * 32;   // this wave's dims
  half_t* const xf = reinterpret_cast<half_t*>(smem_raw) + wave * (RB * SB * 512) + lane * 8;  // its fragments of X
  unsigned char* const regions = smem_raw + S::X_BYTES;
  float* const zpart = reinterpret_cast<float*>(regions + wave * S::REGION) + lane * 4;
  half_t* const stage = reinterpret_cast<half_t*>(regions + wave * S::REGION);
  half_t* const gs = reinterpret_cast<half_t*>(regions + NW * S::REGION);
  uint32_t* const mask = reinterpret_cast<uint32_t*>(regions + NW * S::REGION + S::G_BYTES);  // [2][P][32], by tile parity

  // Which label of a tile (of block lb) and which of the wave's dims a lane's s-th piece of weights and momentum holds.
  constexpr bool LINES = S::LINES;
  [[maybe_unused]] const int low = i & 7, second = i >> 3;
  auto label_of = [&](int lb, int s) { return LINES ? 16 * lb + 8 * (s & 1) + low : 16 * lb + i; };
  auto col_of = [&](int s) { return (LINES ? 32 * ((s & ~1) + second) : 32 * s) + 8 * g; };
  auto at_stage = [&](int lb, int s) { return (LINES ? (s & ~1) + second : s) * 1024 + label_of(lb, s) * 32 + 8 * g; };
  // the first tile's weights; then everything that is set up once while they are on their way
  half8 wcur[2][SB], wnext[2][SB];
  [[maybe_unused]] half8 m[2][SB], mnext[2][SB];
  auto load = [&](const half_t* base, int64_t ld, int tile, half8 (&v)[2][SB]) {
#pragma unroll
    for (int lb = 0; lb < 2; ++lb) {
#pragma unroll
      for (int s = 0; s < SB; ++s) {
        const int label = tile * 32 + label_of(lb, s);
        const half8* p = reinterpret_cast<const half8*>(base + (int64_t)(label < a.L ? label : a.L - 1) * ld + dim0 + col_of(s));
        if constexpr (LINES) v[lb][s] = __builtin_nontemporal_load(p);
        else v[lb][s] = *p;
      }
    }
  };
  half8 xv[P][SB][2];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int s = 0; s < SB; ++s)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int row = 32 * p + 8 * (i >> 2) + 4 * b + (i & 3);
        xv[p][s][b] = *reinterpret_cast<const half8*>(a.X + (int64_t)(row < a.B ? row : a.B - 1) * a.ldx + dim0 + 32 * s + 8 * g);
      }
  load(a.W, a.ldw, blockIdx.x, wcur);
  if constexpr (AHEAD && STEP) load(a.Mo, a.ldm, blockIdx.x, m);

  // label pairs, a few per thread, kept for all tiles (label -1: none, or out of range)
  int plab[S::PAIRS], prow[S::PAIRS];
#pragma unroll
  for (int e = 0; e < S::PAIRS; ++e) {
    const int p = tid + e * S::NT;
    int64_t r = -1, c = -1;
    if (e * S::NT < a.nnz && p < a.nnz) {  // (the first is uniform)
      if (a.pos_x) {
        r = a.pos_x[p];
        c = a.pos_y[p];
      } else if (p >= a.rowptr[0] && p < a.rowptr[a.B]) {
        c = a.colidx[p];
        int lo = 0, hi = a.B - 1;  // the row is the first b with rowptr[b + 1] > p
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (a.rowptr[mid + 1] > p) hi = mid;
          else lo = mid + 1;
        }
        r = lo;
      }
    }
    const bool in = r >= 0 && r < a.B && c >= 0 && c < a.L;
    plab[e] = in ? (int)c : -1;
    prow[e] = in ? (int)r : 0;
  }
  for (int w = tid; w < 2 * S::MASK_WORDS; w += S::NT) mask[w] = 0u;

  // Rows past the batch: zeros for dW, so that they add nothing; the last row again for z.  Zeros there too would make z of
  // a label with an infinite weight no number, hence G, and dW in all dims of that label (0 . NaN); this way G holds
  // nothing there that it does not hold for a row of the batch.
  [[maybe_unused]] half8 xt[P][SB][2];  // A side of dW: dim 8 (i / 4) + 4 b + i % 4, rows 8 g ..+7
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int s = 0; s < SB; ++s) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int rel = 8 * (i >> 2) + 4 * b + (i & 3), row = 32 * p + rel;
        half8 v = xv[p][s][b];
        *reinterpret_cast<half8*>(xf + ((p * 2 + b) * SB + s) * 512) = v;
        if constexpr (STEP) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = row < a.B ? v[e] : (half_t)0.f;
          *reinterpret_cast<half8*>(stage + rel * 32 + 8 * g) = v;
        }
      }
      if constexpr (STEP) {
        S::lds_done();
#pragma unroll
        for (int b = 0; b < 2; ++b) xt[p][s][b] = S::read_tr(stage, t4, 8 * (lane & 3) + 4 * b);
        S::lds_done();
      }
    }
  [[maybe_unused]] float4v acc[RB][SB][2];
  if constexpr (STEP) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int s = 0; s < SB; ++s) acc[rb][s][0] = acc[rb][s][1] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  S::barrier();  // the masks are clear

  int parity = 0;
  for (int tile = blockIdx.x; tile < a.tiles; tile += gridDim.x, parity ^= 1) {
    const int l0 = tile * 32;
    if (l0 + 32 > a.L) {  // labels past the last one weigh nothing (their loads repeated the last label)
#pragma unroll
      for (int lb = 0; lb < 2; ++lb)
#pragma unroll
        for (int s = 0; s < SB; ++s)
#pragma unroll
          for (int e = 0; e < 8; ++e) wcur[lb][s][e] = l0 + label_of(lb, s) < a.L ? wcur[lb][s][e] : (half_t)0.f;
    }
    const int next = tile + (int)gridDim.x;
    if constexpr (AHEAD) {
      if (next < a.tiles) {
        load(a.W, a.ldw, next, wnext);
        if constexpr (STEP) load(a.Mo, a.ldm, next, mnext);
      }
    }
    uint32_t* const mk = mask + parity * S::MASK_WORDS;
#pragma unroll
    for (int e = 0; e < S::PAIRS; ++e) {
      const uint32_t off = (uint32_t)(plab[e] - l0);
      if (plab[e] >= 0 && off < 32u) atomicOr(&mk[(prow[e] >> 5) * 32 + off], 1u << (prow[e] & 31));
    }

    // z, this wave's dims
    {
      float4v z[RB][2];
#pragma unroll
      for (int r = 0; r < RB; ++r) z[r][0] = z[r][1] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < SB; ++s) {
        half8 w[2];  // the B side: label 16 lb + i, dims 32 s + 8 g ..+7
#pragma unroll
        for (int lb = 0; lb < 2; ++lb) {
          w[lb] = wcur[lb][s];
          if constexpr (LINES) w[lb] = S::pick(second == (s & 1), w[lb], S::across8(wcur[lb][s ^ 1]));
        }
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const half8 x = *reinterpret_cast<const half8*>(xf + (r * SB + s) * 512);
#pragma unroll
          for (int lb = 0; lb < 2; ++lb) z[r][lb] = S::mfma(x, w[lb], z[r][lb]);
          if constexpr (!AHEAD) { if (r & 1) __builtin_amdgcn_sched_barrier(0); }  // reads moved up cost spills
        }
      }
      float4v own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < S::UNITS; ++u) {  // u = (p, b, lb)
        if (S::SKIP && u == wave) own = z[u >> 1][u & 1];
        else *reinterpret_cast<float4v*>(zpart + (S::SKIP && u > wave ? u - 1 : u) * 256) = z[u >> 1][u & 1];
      }
      if constexpr (!AHEAD && STEP) load(a.Mo, a.ldm, tile, m);
      S::barrier();
#pragma unroll
      for (int uu = 0; uu < (S::UNITS + NW - 1) / NW; ++uu) {
        const int u = wave + uu * NW;
        if (u < S::UNITS) {
          float4v t = own;
#pragma unroll
          for (int w = 0; w < NW; ++w) {
            const float* zp = reinterpret_cast<const float*>(regions + w * S::REGION) + lane * 4;
            if (!S::SKIP) t += *reinterpret_cast<const float4v*>(zp + u * 256);
            else if (w != wave) t += *reinterpret_cast<const float4v*>(zp + (u > w ? u - 1 : u) * 256);
          }
          const int p = u >> 2, b = (u >> 1) & 1, lb = u & 1;
          const int label = 16 * lb + i, row = 32 * p + 8 * g + 4 * b;
          const uint32_t bits = mk[p * 32 + label] >> (8 * g + 4 * b);
          const bool in = l0 + label < a.L;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float v = sigmoidf_fast(t[r]);
            if ((bits >> r) & 1u) v -= 1.0f;
            gs[(row + r) * 32 + label] = in ? (half_t)v : (half_t)0.f;
          }
        }
      }
    }
    // the next tile's masks: last read before the barrier above, next written past the one below
    for (int w = tid; w < S::MASK_WORDS; w += S::NT) mask[(parity ^ 1) * S::MASK_WORDS + w] = 0u;
    S::barrier();

    if constexpr (!STEP) {  // (every wave has its part of z read before the barrier above)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
        if (wave == rb && 16 * rb + i < a.B && l0 + 8 * g < a.n_store)
          *reinterpret_cast<half8*>(a.G + (int64_t)(16 * rb + i) * a.ldg + l0 + 8 * g) =
              *reinterpret_cast<const half8*>(gs + (16 * rb + i) * 32 + 8 * g);
#pragma unroll
      for (int lb = 0; lb < 2; ++lb)
#pragma unroll
        for (int s = 0; s < SB; ++s) wcur[lb][s] = wnext[lb][s];
      continue;
    }
    // dX^T += W^T . G^T; the waves' regions are their own again
#pragma unroll
    for (int s = 0; s < SB; ++s)
#pragma unroll
      for (int lb = 0; lb < 2; ++lb) *reinterpret_cast<half8*>(stage + at_stage(lb, s)) = wcur[lb][s];
    if constexpr (!AHEAD) {
      if (next < a.tiles) load(a.W, a.ldw, next, wcur);
    }
    {
      half8 bg[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        bg[rb] = *reinterpret_cast<const half8*>(gs + (16 * rb + i) * 32 + 8 * g);
        if (wave == rb && 16 * rb + i < a.B && l0 + 8 * g < a.n_store)
          *reinterpret_cast<half8*>(a.G + (int64_t)(16 * rb + i) * a.ldg + l0 + 8 * g) = bg[rb];
      }
      S::lds_done();
#pragma unroll
      for (int s = 0; s < SB; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const half8 wt = S::read_tr(stage + s * 1024, t4, 16 * c + 4 * (lane & 3));
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) acc[rb][s][c] = S::mfma(wt, bg[rb], acc[rb][s][c]);
          if constexpr (!AHEAD) { if (c) __builtin_amdgcn_sched_barrier(0); }
        }
    }

    // dW^T = X^T . G^T and the update, in the registers that hold the weights
#pragma unroll
    for (int lb = 0; lb < 2; ++lb) {
      half8 gt[P];
#pragma unroll
      for (int p = 0; p < P; ++p) gt[p] = S::read_tr(gs + p * 1024, t4, 16 * lb + 4 * (lane & 3));
      auto product = [&](int s, float4v (&dw)[2]) {  // label 16 lb + i, dims 32 s + 8 g ..+7
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          dw[b] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int p = 0; p < P; ++p) dw[b] = S::mfma(xt[p][s][b], gt[p], dw[b]);
        }
      };
      auto update = [&](int s, const float4v (&dw)[2]) {  // a lane's s-th piece
        half8 wv = wcur[lb][s], mv = m[lb][s];
        if constexpr (!AHEAD) wv = *reinterpret_cast<const half8*>(stage + at_stage(lb, s));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float wf = (float)wv[e];
          const float gg = dw[e >> 2][e & 3] + a.wd * wf;
          const float mf = a.mu * (float)mv[e] + gg;
          mv[e] = (half_t)mf;
          wv[e] = (half_t)(wf - a.lr * mf);
        }
        const int label = l0 + label_of(lb, s);
        if (label < a.L) {
          store<S::LINES ? PAST : CACHED>(reinterpret_cast<half8*>(a.Mo + (int64_t)label * a.ldm + dim0 + col_of(s)), mv);
          store<S::LINES ? PAST : CACHED>(reinterpret_cast<half8*>(a.W + (int64_t)label * a.ldw + dim0 + col_of(s)), wv);
        }
        if constexpr (!AHEAD) __builtin_amdgcn_sched_barrier(0);
      };
      if constexpr (LINES) {
#pragma unroll
        for (int s = 0; s < SB; s += 2) {
          float4v dw[2][2], mine[2];
          product(s, dw[0]);
          product(s + 1, dw[1]);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int b = 0; b < 2; ++b) mine[b] = S::pick(second == h, dw[h][b], S::across8(dw[1 - h][b]));
            update(s + h, mine);
          }
        }
      } else {
#pragma unroll
        for (int s = 0; s < SB; ++s) {
          float4v dw[2];
          product(s, dw);
          update(s, dw);
        }
      }
    }
    if constexpr (AHEAD) {
#pragma unroll
      for (int lb = 0; lb < 2; ++lb)
#pragma unroll
        for (int s = 0; s < SB; ++s) { wcur[lb][s] = wnext[lb][s]; m[lb][s] = mnext[lb][s]; }
    }
    S::lds_done();  // the reads of the region are over before the next tile's parts of z go there
  }

  if constexpr (!STEP) return;
  float* const part = a.part + (int64_t)blockIdx.x * a.B * D;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int row = 16 * rb + i;
    if (row < a.B) {
#pragma unroll
      for (int s = 0; s < SB; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          *reinterpret_cast<float4v*>(part + (int64_t)row * D + dim0 + 32 * s + 16 * c + 4 * g) = acc[rb][s][c];
    }
  }
}

}  // namespace xfc
