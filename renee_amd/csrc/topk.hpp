// Top-K labels per row of X . W^T for K <= 8: the scores are formed once and only the largest of every block of
// consecutive labels is kept; a second kernel picks each row's K best blocks and forms their scores again.
//
// Why that is exact.  Order a row's labels by score descending and label ascending, and its blocks by their best label
// in that order (the block's maximum descending, block ascending: blocks are ranges of labels).  A label among the K best
// lies in one of the K best blocks, because every block ahead of its own holds a label ahead of it.  The second kernel's
// scores are the first one's to the last bit (the same MFMAs in the same order), so a tie is a tie in both.
//
// What it replaced, but where these stay the faster (topk_lists.hpp): lists of the K best kept per workgroup in the LDS beside a
// ring of two slots, a filter against shared bounds in every tile's epilogue and exact retakes of the tiles that overflowed it,
// then a merge of the lists.  Here an epilogue is one maximum per two scores, the ring keeps its third slot, and no tile depends
// on what came before.
#pragma once
#include "pipe_core.hpp"
#include "wide_core.hpp"

namespace xfc {

constexpr int TOPK_MAX = 8;
constexpr int64_t TOPK_RANGE_MAX = (int64_t)1 << 30;  // labels of a range: the kernels' 32-bit indices run somewhat past its end
typedef float float2v __attribute__((ext_vector_type(2)));

// Floats as unsigned keys in the same order, and back.
__device__ __forceinline__ uint32_t topk_key(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float topk_unkey(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
// (score, id) as one number that orders by score descending and id ascending when sorted descending; -0 ranks with +0, and
// a score that is no number ranks below everything (0: no entry).
__device__ __forceinline__ unsigned long long topk_entry(float v, uint32_t id) {
  return v == v ? ((unsigned long long)topk_key(v == 0.f ? 0.f : v) << 32) | (uint32_t)~id : 0ull;
}

// The larger number; an operand that is no number loses.  (Spelled out: the compiler puts an instruction that quiets
// signalling NaNs in front of each operand it knows nothing about, and an MFMA makes none.  Not for what an MFMA has just
// written: the compiler does not count the wait states that inline asm needs.)
__device__ __forceinline__ float max3_num(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float max_num(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// max(a of this lane, a of the lane 32 away) in lanes 0-31, the same of b in lanes 32-63; and 16 away, of every 32.  (Two
// wait states between a vector instruction's result and the exchange, written out for results of inline asm.)
__device__ __forceinline__ float fold32(float a, float b) {
  asm("s_nop 1" : "+v"(a), "+v"(b));
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return max_num(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float fold16(float a, float b) {
  asm("s_nop 1" : "+v"(a), "+v"(b));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return max_num(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

struct ScoreArgs {
  const half_t* X; int64_t ldx;  // M rows of K
  const half_t* W; int64_t ldw;  // N labels of K
  float* bmax; int64_t ldb;      // [M][ldb]: the largest score of every block
  int M, N, K;                   // N at most TOPK_RANGE_MAX
  int tiles_m, tiles_n, n_ids;   // wide: n_ids = tiles_m * round_up(tiles_n, 8)
  int run;                       // small: units in a row that a wave takes, 1, 2 or 4
};

// ---------------------------------------------------------------------------------------------
// more than SCORE_SMALL_ROWS rows, or from the third on with weights that no cache holds: the forward pass's main loop, blocks
// of 32 labels
// ---------------------------------------------------------------------------------------------
// Bound as the forward pass is, by the matrix pipes above 128 rows (1024 rows x 2,812,281 labels x 768: 3.75 ms, 1.18 PFLOP/s; the
// whole call 4.27 -> 3.74 ms) and by the stream of weights on the 128-row tile (65 rows x 700,001 x 768: 195 us, 5.5 TB/s, the whole
// call 341 -> 223 us).  From 33 rows on that tile is as fast as weights streamed past the rows, or faster (64 rows x 700,001 x
// 768: 223 against 243 us, x 4,000: 31 against 35; 32 rows: 223 against 229, x 4,000: 31 against 25).
constexpr int SCORE_WIDE_BLOCK = 32;

using ScoreWide = WideCore<256, 256, 2, 2, true>;
using ScoreWide128 = WideCore<256, 128, 2, 2, true, true>;

template <class C>
__global__ void __launch_bounds__(C::NT) score_wide_kernel(ScoreArgs a) {
  static_assert(C::FM == 8, "a lane holds eight labels of each of four blocks");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* lds = reinterpret_cast<half_t*>(smem_raw);
  const int G = gridDim.x, w = blockIdx.x;
  const int n_items = (a.n_ids - w + G - 1) / G;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN;
  // The row tiles of a label tile side by side on one XCD, as in the forward pass, and an eighth of the label tiles in a row
  // for each XCD, so that the 32 bytes of maxima that a tile has for a row meet their line's other three in its L2.
  auto tile_of = [&](int item, int& mt, int& nt) {
    const int id = item * G + w, xcd = id & 7, local = id >> 3;
    mt = local % a.tiles_m;
    nt = xcd * ((a.tiles_n + 7) >> 3) + local / a.tiles_m;
  };
  auto get = [&](int item, typename C::Operand& oa, typename C::Operand& ob, int& kb, int& ke) {
    int mt, nt;
    tile_of(item, mt, nt);
    oa = typename C::Operand{a.W, a.ldw, nt < a.tiles_n ? nt * C::BM : 0, a.N};
    ob = typename C::Operand{a.X, a.ldx, mt * C::BN, a.M};
    kb = 0;
    ke = a.K;
  };
  auto epilogue = [&](int item, float4v (&acc)[C::FM][C::FN]) {
    int mt, nt;
    tile_of(item, mt, nt);
    if (nt >= a.tiles_n) return;
    const int row_l = mt * C::BN + wn * C::TN + (lane & 15);
    const int col_l = nt * C::BM + wm * C::TM + 8 * (lane >> 4);
    auto body = [&](auto edge_tag) {
      constexpr bool EDGE = decltype(edge_tag)::value;
#pragma unroll
      for (int fn = 0; fn < C::FN; ++fn) {
        float m[4];  // of this lane's eight labels of block p
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const float4v lo = C::value(acc[2 * p][fn]), hi = C::value(acc[2 * p + 1][fn]);
          float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          if constexpr (EDGE) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = col_l + 32 * p + e < a.N ? v[e] : __builtin_nanf("");
          }
          m[p] = max3_num(max3_num(v[0], v[1], v[2]), v[3], max3_num(v[4], v[5], max_num(v[6], v[7])));
        }
        // lanes 16 g .. 16 g + 15 end up with block g of their row
        const float best = fold16(fold32(m[0], m[2]), fold32(m[1], m[3]));
        const int row = row_l + 16 * fn;
        if (row < a.M) a.bmax[(int64_t)row * a.ldb + (nt * C::BM + wm * C::TM) / SCORE_WIDE_BLOCK + (lane >> 4)] = best;
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (nt * C::BM + C::BM > a.N) body(std::true_type{});
    else body(std::false_type{});
  };
  C::run(0, n_items, lds, get, epilogue);
}

// ---------------------------------------------------------------------------------------------
// up to SCORE_SMALL_ROWS rows of weights that the caches hold, two of any: the weights stream past the rows, blocks of 16 labels
// ---------------------------------------------------------------------------------------------
// Bound by the stream of weights.  X lies in the LDS as MFMA fragments, RB blocks of 16 rows; a wave takes units of 16
// labels, loads them straight into the A side's registers (16 rows x 64 bytes an instruction) and keeps two to three
// pieces of SCORE_STEPS loads on their way, across units: a fetch never waits for an epilogue.  Waves never meet.
// 16 rows x 131,072 labels x 768: 37.5 us, 5.4 TB/s; the whole call 108 -> 57 us.  At 700,001 labels the stores of the maxima
// (a row's lie apart, a few bytes each) are 25 of 206 us.
constexpr int SCORE_SMALL_ROWS = 32, SCORE_SMALL_BLOCK = 16, SCORE_SMALL_WAVES = 8, SCORE_STEPS = 4, SCORE_SLOTS = 3;

template <int RB>
constexpr int64_t score_small_lds(int64_t K) { return (K + 31) / 32 * RB * 1024; }

// Two workgroups to a CU.
template <int RB>
__global__ void __launch_bounds__(64 * SCORE_SMALL_WAVES, 4) score_small_kernel(ScoreArgs a) {
  constexpr int NW = SCORE_SMALL_WAVES;
  static_assert(RB <= 4, "a lane stores the maxima of one row");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* const xs = reinterpret_cast<half_t*>(smem_raw);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int n_units = (a.N + SCORE_SMALL_BLOCK - 1) / SCORE_SMALL_BLOCK, nk = (a.K + 31) / 32;
  const int pieces = (nk + SCORE_STEPS - 1) / SCORE_STEPS;  // of a unit
  const int run = a.run, skip = (int)(gridDim.x * NW - 1) * run + 1;  // from the last unit of a run to the first of the next
  auto next = [&](int u) { return (u + 1) & (run - 1) ? u + 1 : u + skip; };
  // Neighbouring workgroups of an XCD take neighbouring units: the units of a line of maxima meet in one L2.
  const int eighth = gridDim.x >> 3, block = (gridDim.x & 7) == 0 ? (blockIdx.x & 7) * eighth + (blockIdx.x >> 3) : blockIdx.x;
  int unit = (block * NW + wave) * run;

  // Fetch cursor.  Past the last unit it repeats that one, so that the number of loads on their way is always the same.
  int f_unit = unit < n_units ? unit : n_units - 1, f_piece = 0;
  half8 w[SCORE_SLOTS][SCORE_STEPS];
  const half_t* row = nullptr;
  auto open = [&]() {
    const int label = f_unit * SCORE_SMALL_BLOCK + i;
    row = a.W + (int64_t)(label < a.N ? label : a.N - 1) * a.ldw;
  };
  open();
  auto fetch = [&](half8 (&dst)[SCORE_STEPS]) {
#pragma unroll
    for (int j = 0; j < SCORE_STEPS; ++j) {
      const int k = (f_piece * SCORE_STEPS + j) * 32 + 8 * g;  // past K: any k, multiplied by nothing or cleared below
      dst[j] = *reinterpret_cast<const half8*>(row + (k < a.K ? k : 0));
    }
    if (++f_piece == pieces) {
      f_piece = 0;
      if (next(f_unit) < n_units) f_unit = next(f_unit);
      open();
    }
  };
#pragma unroll
  for (int s = 0; s < SCORE_SLOTS; ++s) fetch(w[s]);

  for (int q = threadIdx.x; q < nk * RB * 64; q += 64 * NW) {
    const int l = q & 63, rb = (q >> 6) % RB, s = (q >> 6) / RB;
    const int r = 16 * rb + (l & 15), k = 32 * s + 8 * (l >> 4);
    half8 v = {};
    if (r < a.M && k < a.K) v = *reinterpret_cast<const half8*>(a.X + (int64_t)r * a.ldx + k);
    *reinterpret_cast<half8*>(xs + q * 8) = v;
  }
  __syncthreads();

  float4v z[RB], best[RB];
  int piece = 0;
  while (unit < n_units) {
#pragma unroll
    for (int s = 0; s < SCORE_SLOTS; ++s) {
      if (unit < n_units) {
        if (piece == 0) {
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) z[rb] = float4v{0.f, 0.f, 0.f, 0.f};
        }
        const half_t* const xp = xs + (piece * SCORE_STEPS * RB * 64 + lane) * 8;
        auto step = [&](int j, const half8& wv) {
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
            z[rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv, *reinterpret_cast<const half8*>(xp + (j * RB + rb) * 512), z[rb], 0, 0, 0);
        };
        if ((piece + 1) * SCORE_STEPS * 32 <= a.K) {  // no branches: the reads of a step go under the MFMAs before it
#pragma unroll
          for (int j = 0; j < SCORE_STEPS; ++j) step(j, w[s][j]);
        } else {
#pragma unroll
          for (int j = 0; j < SCORE_STEPS; ++j) {
            const int k = (piece * SCORE_STEPS + j) * 32;
            if (k < a.K) {
              half8 wv = w[s][j];
#pragma unroll
              for (int e = 0; e < 8; ++e) wv[e] = k + 8 * g < a.K ? wv[e] : (half_t)0.f;
              step(j, wv);
            }
          }
        }
        if (++piece == pieces) {
          piece = 0;
          const int r4 = unit & (run - 1);
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) {
            if ((unit + 1) * SCORE_SMALL_BLOCK > a.N) {
#pragma unroll
              for (int r = 0; r < 4; ++r) z[rb][r] = unit * SCORE_SMALL_BLOCK + 4 * g + r < a.N ? z[rb][r] : __builtin_nanf("");
            }
            float m = fmaxf(fmaxf(z[rb][0], z[rb][1]), fmaxf(z[rb][2], z[rb][3]));
            m = fold32(m, m);
            m = fold16(m, m);
#pragma unroll
            for (int r = 0; r < 4; ++r) best[rb][r] = r4 == r ? m : best[rb][r];
          }
          const int after = next(unit);
          if (after != unit + 1 || run == 1 || after >= n_units) {
            float4v out = best[0];  // lanes 16 g .. 16 g + 15 store the rows of block g
#pragma unroll
            for (int rb = 1; rb < RB; ++rb) out = g == rb ? best[rb] : out;
            if (g < RB && 16 * g + i < a.M) {
              float* const dst = a.bmax + (int64_t)(16 * g + i) * a.ldb + (unit - r4);
              if (run == 4) *reinterpret_cast<float4v*>(dst) = out;
              else if (run == 2) *reinterpret_cast<float2v*>(dst) = float2v{out[0], out[1]};
              else *dst = out[0];
            }
          }
          unit = after;
        }
      }
      fetch(w[s]);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// the K best blocks of each row, their scores, the K best of those
// ---------------------------------------------------------------------------------------------
struct PickArgs {
  const half_t* X; int64_t ldx;
  const half_t* W; int64_t ldw;
  const float* bmax; int64_t ldb;  // ldb a multiple of 4
  int n_blocks;                    // of this range of labels
  int N, K;                        // its labels (W points at the first), feature dims
  int64_t first;                   // id of its first label
  int topk;
  unsigned long long* best;        // [rows][topk]: the K best of the ranges before, and what this one leaves; null: one range
  int begin, end;                  // the first range, the last
  int64_t numy;
  float* out_v; int64_t* out_i;
};

// The largest of the wave's 32-bit numbers, uniform: within rows of 16 lanes, then across them.
__device__ __forceinline__ uint32_t wave_max32(uint32_t v) {
  auto step = [&](auto ctrl, auto rows) {
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, decltype(rows)::value, 0xf, true);
    v = o > v ? o : v;
  };
  using std::integral_constant;
  step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});  // row_shr:1, 2, 4, 8
  step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});
  step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});
  step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});
  step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});  // row_bcast:15, 31
  step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// The same of 64-bit keys, uniform: by their upper halves, and by the lower ones of those that share the largest, if there are
// several.  (By shuffles of whole keys, six steps through the LDS, topk_pick_kernel took 23.6 us at 16 x 131,072 and K = 5, then 14.)
__device__ __forceinline__ unsigned long long wave_max(unsigned long long k) {
  const uint32_t hi = wave_max32((uint32_t)(k >> 32));
  const unsigned long long with = __ballot((uint32_t)(k >> 32) == hi);
  uint32_t lo;
  if ((with & (with - 1)) == 0) lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, __builtin_ctzll(with));
  else lo = wave_max32((uint32_t)(k >> 32) == hi ? (uint32_t)k : 0u);
  return ((unsigned long long)hi << 32) | lo;
}
// The K largest of the wave's keys, all different but for 0, in lanes 0 .. K - 1 (0 where there are fewer).
__device__ __forceinline__ unsigned long long wave_top(unsigned long long key, int K, int lane) {
  unsigned long long top = 0;
  if (__ballot(key != 0) == 0) return top;
  for (int r = 0; r < K; ++r) {
    const unsigned long long m = wave_max(key);
    if (m == 0) break;
    if (lane == r) top = m;
    if (key == m) key = 0;
  }
  return top;
}

// One workgroup per row.  With few blocks or many rows bound by its instructions (25 us at 700 rows x 282 blocks, where seven of
// a thread's eight fetches brought nothing and six of the eight waves put zeros in order): what has nothing to do is left out.  Else by reading the blocks' maxima and the chosen blocks' weights (1024 rows x 87,885 blocks, K = 5: 122 us,
// 5 TB/s), on small batches by latency (16 x 8,192 blocks: 14 us): each thread finds the best of its blocks,
// the K best threads are looked at again block by block (a wave each), and the K best blocks' scores are formed by MFMAs
// that hold the row in all sixteen columns.  Keys are (score, id) as topk_entry makes them, all different but for 0.
template <int BLOCK>
__global__ void __launch_bounds__(512) topk_pick_kernel(PickArgs a) {
  constexpr int NW = 8, LISTS = NW * TOPK_MAX;
  constexpr int FETCH = 8, STEPS = 8;  // loads on their way: maxima, pieces of the weights
  static_assert(TOPK_MAX * BLOCK <= 512 - TOPK_MAX, "one candidate per thread");
  __shared__ unsigned long long list[LISTS], chosen[TOPK_MAX], kept[TOPK_MAX];
  __shared__ float score[TOPK_MAX * BLOCK];
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.topk;
  const float* maxima = a.bmax + (int64_t)row * a.ldb;
  const int quads = (a.n_blocks + 3) / 4;
  // (a row's maxima are less than 2^32 bytes: a lane keeps one offset per load)
  auto quad = [&](int q) { return *reinterpret_cast<const float4v*>(reinterpret_cast<const char*>(maxima) + 16u * (uint32_t)(q < quads ? q : quads - 1)); };
  // the best key below `bound` of blocks 4 q ..+3, whose maxima are v
  auto best_of = [&](int q, const float4v& v, unsigned long long bound) {
    unsigned long long best = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned long long k = 4 * q + e < a.n_blocks ? topk_entry(v[e], (uint32_t)(4 * q + e)) : 0ull;
      if (k < bound && k > best) best = k;
    }
    return best;
  };
  // out[0..K) = the K largest of the workgroup's keys, in order; all threads of the workgroup call it
  auto top_of_all = [&](unsigned long long key, unsigned long long* out) {
    __syncthreads();
    const unsigned long long own = wave_top(key, K, lane);
    if (lane < K) list[wave * TOPK_MAX + lane] = own;
    __syncthreads();
    if (wave == 0) {
      const unsigned long long top = wave_top((lane & (TOPK_MAX - 1)) < K ? list[lane] : 0ull, K, lane);
      if (lane < K) out[lane] = top;
    }
    __syncthreads();
  };

  if (tid < TOPK_MAX) kept[tid] = a.best && !a.begin && tid < K ? a.best[(int64_t)row * K + tid] : 0ull;
  unsigned long long bound = ~0ull;  // blocks at or above it have been taken
  for (;;) {
    unsigned long long mine = 0;
    for (int q = tid; q - lane < quads; q += 512 * FETCH) {
      const int n = (quads - (q - lane) + 511) / 512;  // of the wave's fetches, those that bring anything new
      float4v v[FETCH];
#pragma unroll
      for (int f = 0; f < FETCH; ++f) v[f] = quad(q + 512 * f);
#pragma unroll
      for (int f = 0; f < FETCH; ++f) {
        if (f >= n) break;
        const unsigned long long k = best_of(q + 512 * f, v[f], bound);
        mine = k > mine ? k : mine;
      }
    }
    top_of_all(mine, chosen);
    // The K best blocks are among those of these K threads, at or above the last of their bests.  Wave w takes thread w's:
    // thread t's quads are t, t + 512, ...
    const unsigned long long head = chosen[wave < K ? wave : 0], least = chosen[K - 1];
    unsigned long long mykey = 0;  // the wave's r-th best, in lane r
    if (wave < K && head != 0) {
      const int first = (int)((~(uint32_t)head / 4) & 511u);
      unsigned long long below = bound, k = 0;
      const int q0 = first + 512 * lane;  // a lane's first quad stays in its registers; there are more above 131,072 blocks
      const float4v v0 = quad(q0);
      auto rescan = [&]() {
        k = best_of(q0, v0, below);
        for (int q = q0 + 512 * 64; q < quads; q += 512 * 64) {
          const unsigned long long c = best_of(q, quad(q), below);
          k = c > k ? c : k;
        }
      };
      rescan();
      for (int r = 0; r < K; ++r) {
        const unsigned long long m = wave_max(k);
        if (m < least || m == 0) break;
        if (lane == r) mykey = m;
        if (k == m) { below = m; rescan(); }
      }
    }
    top_of_all(mykey, chosen);

    int n_sel = 0;
    for (int r = 0; r < K; ++r) n_sel += chosen[r] != 0;
    n_sel = __builtin_amdgcn_readfirstlane(n_sel);
    // their scores, 16 labels at a time; the MFMAs and their order are those of the kernels above
    for (int u = wave; u < n_sel * (BLOCK / 16); u += NW) {
      const int label = (int)~(uint32_t)chosen[u / (BLOCK / 16)] * BLOCK + (u % (BLOCK / 16)) * 16;
      const int mine_l = label + (lane & 15), k8 = 8 * (lane >> 4);
      const half_t* wp = a.W + (int64_t)(mine_l < a.N ? mine_l : a.N - 1) * a.ldw;
      const half_t* xp = a.X + (int64_t)row * a.ldx;
      float4v z = {0.f, 0.f, 0.f, 0.f};
      for (int k0 = 0; k0 < a.K; k0 += 32 * STEPS) {
        half8 wv[STEPS], xv[STEPS];
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
          const int k = k0 + 32 * j + k8;
          wv[j] = *reinterpret_cast<const half8*>(wp + (k < a.K ? k : 0));
          xv[j] = *reinterpret_cast<const half8*>(xp + (k < a.K ? k : 0));
        }
#pragma unroll
        for (int j = 0; j < STEPS; ++j) {
          if (k0 + 32 * j >= a.K) break;
          if (k0 + 32 * j + 32 > a.K) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              wv[j][e] = k0 + 32 * j + k8 < a.K ? wv[j][e] : (half_t)0.f;
              xv[j][e] = k0 + 32 * j + k8 < a.K ? xv[j][e] : (half_t)0.f;
            }
          }
          z = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[j], xv[j], z, 0, 0, 0);
        }
      }
      if ((lane & 15) == 0) *reinterpret_cast<float4v*>(&score[u * 16 + 4 * (lane >> 4)]) = z;
    }
    __syncthreads();
    // the K best of the blocks' labels and of what was there before
    unsigned long long key = 0;
    if (tid < n_sel * BLOCK) {
      const int64_t label = (int64_t)(int)~(uint32_t)chosen[tid / BLOCK] * BLOCK + tid % BLOCK;
      if (label < a.N) key = topk_entry(score[tid], (uint32_t)(a.first + label));
    } else if (tid >= 512 - TOPK_MAX) {
      key = kept[tid - (512 - TOPK_MAX)];
    }
    bound = chosen[K - 1];
    top_of_all(key, kept);
    // (a block whose maximum is -inf may hold nothing but scores that are no numbers: then there may be more elsewhere)
    if (kept[K - 1] != 0 || bound == 0) break;
  }
  if (tid < K) {
    const unsigned long long k = kept[tid];
    if (a.best && !a.end) {
      a.best[(int64_t)row * K + tid] = k;
    } else {
      const int64_t id = k ? (int64_t)(uint32_t)~(uint32_t)k : a.numy;
      a.out_v[(int64_t)row * K + tid] = k ? topk_unkey((uint32_t)(k >> 32)) : -__builtin_huge_valf();
      a.out_i[(int64_t)row * K + tid] = id < a.numy ? id : a.numy - 1;  // padded labels are clamped, as the reference does
    }
  }
}

}  // namespace xfc
