// XFC layer step kernels for gfx950 and their C-ABI entry points.
//
//   fwd   : G = fp16( sigmoid(X . W^T) - Y )      Y subtracted pair by pair after the product
//   dx    : dX = scale * G . W                    split over labels, fp32 partials + reduce
//   dw    : dW = G^T . X, consumed in the tile by  M = mu*M + dW + wd*W ; W -= lr*M
// plus the plain six-argument GEMM the reference extension exposes.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include <atomic>

#include <type_traits>

#include "../../include/xfc_mi355x.h"
#include "back_step.hpp"
#include "back_wide.hpp"
#include "pipe_core.hpp"
#include "small_step.hpp"
#include "tile_plan.hpp"
#include "topk.hpp"
#include "topk_lists.hpp"
#include "wide_core.hpp"

namespace xfc {

// ---------------------------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------------------------
// Workgroup ids are dealt round-robin to the 8 XCDs, each with its own L2.  Tiles that
// share an operand slice are given ids that land on one XCD next to each other:
// id -> (inner, outer) with `inner` (size n_inner) varying fastest among ids of one XCD.
__device__ __forceinline__ void xcd_map(int id, int n_inner, int& inner, int& outer) {
  const int xcd = id & 7, local = id >> 3;
  inner = local % n_inner;
  outer = (local / n_inner) * 8 + xcd;
}

// ---------------------------------------------------------------------------------------------
// forward: out = epilogue(alpha * X . W^T + beta * out)
// ---------------------------------------------------------------------------------------------
enum FwdMode { FWD_LINEAR = 0, FWD_SIGMOID = 1, FWD_SIGMOID_PLAIN = 2 };  // PLAIN: alpha 1, beta 0

// Batches above 128 rows, as a rule: 256 labels (the A side, contiguous in the output) x 256 rows, W running ahead.
using FwdWide = WideCore<256, 256, 2, 2, true>;
static_assert(FwdWide::LDS_BYTES <= 160 * 1024, "LDS budget");
// The same loop on 128 labels x 128 rows, two workgroups to a CU (see fwd_plan).
using FwdWide128 = WideCore<128, 128, 2, 2, true>;
static_assert(2 * FwdWide128::LDS_BYTES <= 160 * 1024, "two to a CU");
template <class C, FwdTile T>
constexpr bool planned = C::BM == fwd_tile_labels(T) && C::BN == fwd_tile_rows(T) && C::BK == FWD_STAGE;
static_assert(planned<FwdWide, FWD_WIDE> && planned<FwdWide128, FWD_WIDE128>, "tile_plan.hpp");
// Batches of up to 128 and 64 rows (the reference's B = 32 plumbing case, --accum micro-batches, the last partial batch
// of an epoch), where a 256-row tile would spend most of its MFMAs on padding: W streams from HBM, eight waves, three
// ring slots.
using FwdCore = PipeCore<128, 256, 64, 2, 4, 3, true, true, false, false, false, 4>;  // one wave per SIMD fetches
using FwdCore64 = PipeCore<64, 256, 64, 2, 4, 3, true, true, false, false, false, 4>;
// beside the ring: store staging (8 rows x TN labels per wave)
template <class C>
struct FwdLds {
  static constexpr int STG_HALVES = 8 * C::TN;
  static constexpr int BYTES = C::LDS_BYTES + C::NW * STG_HALVES * 2;
  static_assert(C::FN % 2 == 0, "staging read-back walks 64-label pieces");
  static_assert(BYTES <= 160 * 1024, "LDS budget");
};
static_assert(FwdCore::BN == fwd_tile_labels(FWD_128) && FwdCore::BM == fwd_tile_rows(FWD_128) && FwdCore64::BN == fwd_tile_labels(FWD_64) &&
              FwdCore64::BM == fwd_tile_rows(FWD_64), "tile_plan.hpp");

constexpr int LOGIT_BLOCK = 32;
// max of two packed halves each, and of three; an operand that is no number wins, so that a block with one can be told.
// (Two wait states in front of the lane exchanges below, as for fold32.)
__device__ __forceinline__ uint32_t pk_max(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_pk_maximum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ uint32_t pk_max(const half8& v) {
  const uint4v q = __builtin_bit_cast(uint4v, v);
  return pk_max(pk_max(q[0], q[1], q[2]), q[3], q[3]);
}
__device__ __forceinline__ uint32_t pk_fold32(uint32_t a, uint32_t b) {
  asm("s_nop 1" : "+v"(a), "+v"(b));
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  return pk_max(r[0], r[1], r[1]);
}
__device__ __forceinline__ uint32_t pk_fold16(uint32_t a, uint32_t b) {
  asm("s_nop 1" : "+v"(a), "+v"(b));
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  return pk_max(r[0], r[1], r[1]);
}
__device__ __forceinline__ half_t pk_larger(uint32_t a) {  // of the two halves
  const uint16_t h = (uint16_t)pk_max(a, a >> 16, a >> 16);
  return __builtin_bit_cast(half_t, h);
}

struct FwdArgs {
  const half_t* X; int64_t ldx;     // M x K, K-contiguous
  const half_t* W; int64_t ldw;     // N x K, K-contiguous
  half_t* out; int64_t ldo;         // M x n_store, row-major
  int M, N, K, n_store;             // columns N <= c < n_store are written as zero
  float alpha, beta;
  double* loss_part; int loss_have; // LOSS: one partial sum per workgroup, the first loss_have added to what is there
  half_t* bmax; int64_t ldb;        // BMAX: [M][ldb] the largest stored value of every LOGIT_BLOCK columns
  int tiles_m, tiles_n, n_ids;      // n_ids = tiles_m * round_up(tiles_n, 8)
  bool through;                     // out is stored through the L2 (see launch_fwd)
};

// Persistent: workgroup w takes tile ids w, w + gridDim.x, ... (gridDim.x a multiple of 8, so an
// id keeps its XCD and the row tiles of one label tile run side by side on one L2).
template <class C, int MODE, bool BETA, bool LOSS = false, bool BMAX = false>
__global__ void __launch_bounds__(C::NT, 160 * 1024 / C::LDS_BYTES) fwd_wide_kernel(FwdArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* lds = reinterpret_cast<half_t*>(smem_raw);
  const int G = gridDim.x, w = blockIdx.x;
  const int n_items = (a.n_ids - w + G - 1) / G;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be
  const int wm = wave / C::WN, wn = wave % C::WN;
  double loss_acc = 0.0;  // LOSS: this lane's share of sum softplus(z)

  auto get = [&](int item, typename C::Operand& oa, typename C::Operand& ob, int& kb, int& ke) {
    int mt, nt;
    xcd_map(item * G + w, a.tiles_m, mt, nt);
    oa = typename C::Operand{a.W, a.ldw, nt < a.tiles_n ? nt * C::BM : 0, a.N};
    ob = typename C::Operand{a.X, a.ldx, mt * C::BN, a.M};
    kb = 0;
    ke = a.K;
  };
  // A lane owns one batch row and eight consecutive labels of every 32: 16-byte stores straight from the registers,
  // 64 bytes per row and instruction, the other 64 of the line with the next.  Of a tile's 54,000 cycles this takes
  // 10,000: the two transcendentals of a sigmoid occupy a SIMD for 32 cycles per 64 elements, which with the conversions
  // is 9,200 (2,900 without the sigmoid), and the stores hide under them; the wait for the last of them to be written
  // was another 1,900 in the next tile's first stage, which now passes them by their count.  Stores of whole lines (8 rows x 128 or 4 x 256 bytes per
  // instruction) take as long: all CUs together store at 7.3 TB/s into the caches whatever the shape.
  auto epilogue = [&](int item, float4v (&acc)[C::FM][C::FN]) {
    int mt, nt;
    xcd_map(item * G + w, a.tiles_m, mt, nt);
    if (nt >= a.tiles_n) return false;
    const int row_l = mt * C::BN + wn * C::TN + (lane & 15);
    const int col_l = nt * C::BM + wm * C::TM + 8 * (lane >> 4);
    // A tile that crosses the label count is compiled as a path of its own: the common one carries no column checks.
    auto body = [&](auto edge_tag) {
      constexpr bool EDGE = decltype(edge_tag)::value;
#pragma unroll
      for (int fn = 0; fn < C::FN; ++fn) {
        const int row = row_l + 16 * fn;
        half_t* dst = a.out + (int64_t)row * a.ldo + col_l;
        const bool row_in = row < a.M;
        [[maybe_unused]] uint32_t largest[C::FM / 2];  // BMAX: of this lane's eight columns of block p
#pragma unroll
        for (int p = 0; p < C::FM / 2; ++p) {
          const int col = col_l + 32 * p;
          const float4v lo = C::value(acc[2 * p][fn]), hi = C::value(acc[2 * p + 1][fn]);
          float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          if constexpr (LOSS) {
            static_assert(MODE == FWD_SIGMOID_PLAIN && !BETA, "the loss is that of the plain logits");
            // softplus(z) = max(z, 0) + log(1 + e^-|z|) (dl_base.py:578-583); the logarithms of a lane's eight factors in
            // (1, 2] are taken as one, of their product.  (With one logarithm per element and the sum formed at the end of
            // the tile the kernel spilled 800 registers: 234 us at 199 x 131,072 x 768, now 84.)
            // The parts are summed apart and in double: of a positive that has been learnt, max(z, 0) goes again with
            // positives_kernel's z and the logarithm is what remains, 4.5e-5 beside 10.
            float prod = 1.f, lin[2] = {0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float t = 1.0f + __builtin_amdgcn_exp2f(fabsf(v[e]) * -1.44269504088896341f);
              const bool in = !EDGE || col + e < a.N;
              prod *= in ? t : 1.f;
              lin[e >> 2] += in ? fmaxf(v[e], 0.f) : 0.f;
            }
            loss_acc += (double)(row_in ? lin[0] : 0.f);
            loss_acc += (double)(row_in ? lin[1] : 0.f);
            loss_acc += (double)(row_in ? 0.69314718056f * __builtin_amdgcn_logf(prod) : 0.f);
            asm volatile("" : "+v"(loss_acc));  // here, not when the tile is done: that would keep every element until then
          }
          if constexpr (BETA) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              v[e] *= a.alpha;
              if (row_in && col + e < a.N) v[e] += a.beta * (float)dst[32 * p + e];
            }
          } else if constexpr (MODE == FWD_SIGMOID) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= a.alpha;
          }
          if constexpr (MODE != FWD_LINEAR) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = sigmoidf_fast(v[e]);
          }
          half8 v8;
#pragma unroll
          for (int e = 0; e < 8; ++e) v8[e] = !EDGE || col + e < a.N ? (half_t)v[e] : (half_t)0.f;
          if (row_in) {
            if (!EDGE || col + 8 <= a.n_store) {
              // (a non-temporal store of half a line is written back before the other half comes: 1.19 against 1.14 ms)
              if (C::FM == 4 && a.through) store<THROUGH>(reinterpret_cast<half8*>(dst + 32 * p), v8);
              else *reinterpret_cast<half8*>(dst + 32 * p) = v8;
            } else {
#pragma unroll
              for (int e = 0; e < 8; ++e)
                if (col + e < a.n_store) dst[32 * p + e] = v8[e];
            }
          }
          if constexpr (BMAX) {
            static_assert(MODE == FWD_LINEAR && (C::FM == 8 || C::FM == 4), "four blocks of logits or two, eight columns of each in a lane");
            half8 m8 = v8;
#pragma unroll
            for (int e = 0; e < 8; ++e) m8[e] = !EDGE || col + e < a.N ? v8[e] : (half_t)-__builtin_huge_valf();
            largest[p] = pk_max(m8);
          }
          __builtin_amdgcn_sched_barrier(0);  // eight elements in flight are enough; more of them spill
        }
        if constexpr (BMAX) {
          // lanes 16 g .. 16 g + 15 end up with block g of their row
          constexpr int BACK = C::FM / 2 - 2;  // (of two blocks the upper half of the lanes holds what the lower does)
          const half_t m = pk_larger(pk_fold16(pk_fold32(largest[0], largest[BACK]), pk_fold32(largest[1], largest[1 + BACK])));
          if (row_in && (lane >> 4) < C::FM / 2) a.bmax[(int64_t)row * a.ldb + (nt * C::BM + wm * C::TM) / LOGIT_BLOCK + (lane >> 4)] = m;
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (nt * C::BM + C::BM > a.N) {
      body(std::true_type{});
      return false;
    }
    body(std::false_type{});
    return mt * C::BN + (wn + 1) * C::TN <= a.M;
  };
  C::template run<C::FN * C::FM / 2>(0, n_items, lds, get, epilogue);
  if constexpr (LOSS) {
    // deterministic: lanes -> wave (butterfly), waves -> workgroup (LDS, fixed order), one partial per workgroup
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss_acc += __shfl_xor(loss_acc, off, 64);
    double* red = reinterpret_cast<double*>(smem_raw);
    __syncthreads();
    if (lane == 0) red[wave] = loss_acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int i = 0; i < C::NW; ++i) t += red[i];
      // (only small tiles come after others; asked of large ones too, their kernel keeps 13 more scalars in vector lanes)
      a.loss_part[w] = C::FM == 4 && w < a.loss_have ? a.loss_part[w] + t : t;
    }
  }
}

// The same on the smaller row tiles.
template <class C, int MODE, bool BETA, bool LOSS = false, bool BMAX = false>
__global__ void __launch_bounds__(C::NT) fwd_kernel(FwdArgs a) {
  constexpr int FWD_STG_HALVES = FwdLds<C>::STG_HALVES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* lds = reinterpret_cast<half_t*>(smem_raw);
  const int G = gridDim.x, w = blockIdx.x;
  const int n_items = (a.n_ids - w + G - 1) / G;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be
  const int wm = wave / C::WN, wn = wave % C::WN;
  half_t* stg = reinterpret_cast<half_t*>(smem_raw + C::LDS_BYTES) + wave * FWD_STG_HALVES;  // 8 rows x TN labels
  double loss_acc = 0.0;  // LOSS: this lane's share of sum softplus(z)

  auto get = [&](int item, typename C::Operand& oa, typename C::Operand& ob, int& kb, int& ke) {
    int mt, nt;
    xcd_map(item * G + w, a.tiles_m, mt, nt);
    oa = typename C::Operand{a.X, a.ldx, mt * C::BM, a.M, a.K};
    ob = typename C::Operand{a.W, a.ldw, nt < a.tiles_n ? nt * C::BN : 0, a.N, a.K};
    kb = 0;
    ke = a.K;
  };
  auto epilogue = [&](int item, float16v (&acc)[C::FM][C::FN]) {
    int mt, nt;
    xcd_map(item * G + w, a.tiles_m, mt, nt);
    if (nt >= a.tiles_n) return;
    const int m0 = mt * C::BM, n0 = nt * C::BN;
    const int h = lane >> 5;
    constexpr int CHS = C::TN / 8;  // 16-byte chunks per staged row
    // A tile that crosses the label count is compiled as a path of its own: the common one carries no column checks.
    int64_t lane_off[C::FN / 2];  // where this lane's 16 bytes of a staged strip go, relative to the strip
#pragma unroll
    for (int p = 0; p < C::FN / 2; ++p) lane_off[p] = (int64_t)((lane + 64 * p) / CHS) * a.ldo + ((lane + 64 * p) % CHS) * 8;
    auto body = [&](auto edge_tag) {
      constexpr bool EDGE = decltype(edge_tag)::value;
      if constexpr (LOSS) {
        static_assert(MODE == FWD_SIGMOID_PLAIN && !BETA, "the loss is that of the plain logits");
        // The loss terms in a pass of their own over the accumulators, one block at a time (see fwd_wide_kernel)
#pragma unroll
        for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
          for (int fn = 0; fn < C::FN; ++fn) {
            const int ecol = n0 + wn * C::TN + fn * 32 + (lane & 31);
            float prod = 1.f, lin = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const float v = acc[fm][fn][r];
              const float t = 1.0f + __builtin_amdgcn_exp2f(fabsf(v) * -1.44269504088896341f);
              const bool in = !EDGE || (m0 + wm * C::TM + fm * 32 + c_row(r, lane) < a.M && ecol < a.N);
              prod *= in ? t : 1.f;
              lin += in ? fmaxf(v, 0.f) : 0.f;
              if ((r & 3) == 3) {
                loss_acc += (double)lin;
                lin = 0.f;
              }
            }
            loss_acc += (double)(0.69314718056f * __builtin_amdgcn_logf(prod));
            asm volatile("" : "+v"(loss_acc));
            __builtin_amdgcn_sched_barrier(0);
          }
      }
#pragma unroll
      for (int fm = 0; fm < C::FM; ++fm) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int fn = 0; fn < C::FN; ++fn) {
            const int ecol = n0 + wn * C::TN + fn * 32 + (lane & 31);
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
              const int r = 4 * q + rr;
              float v = acc[fm][fn][r];
              if constexpr (BETA) {
                v *= a.alpha;
                const int erow = m0 + wm * C::TM + fm * 32 + c_row(r, lane);
                if (erow < a.M && ecol < a.N) v += a.beta * (float)a.out[(int64_t)erow * a.ldo + ecol];
              } else if constexpr (MODE == FWD_SIGMOID) {
                v *= a.alpha;
              }
              if constexpr (MODE != FWD_LINEAR) v = sigmoidf_fast(v);
              if constexpr (EDGE) { if (ecol >= a.N) v = 0.f; }
              stg[(4 * h + rr) * C::TN + fn * 32 + (lane & 31)] = (half_t)v;
            }
          }
          // the wave's LDS traffic is ordered: its own writes above are visible to the reads below
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
#pragma unroll
          for (int p = 0; p < C::FN / 2; ++p) {
            const int cid = lane + 64 * p;
            const int srow = cid / CHS, sch = cid % CHS;
            const half8 v8 = *reinterpret_cast<const half8*>(stg + srow * C::TN + sch * 8);
            const int row = m0 + wm * C::TM + fm * 32 + 8 * q + srow;
            const int col = n0 + wn * C::TN + sch * 8;
            if constexpr (BMAX) {  // four neighbouring lanes hold a block
              static_assert(MODE == FWD_LINEAR && CHS % 4 == 0, "whole blocks of logits in a staged row");
              half8 m8 = v8;
#pragma unroll
              for (int e = 0; e < 8; ++e) m8[e] = !EDGE || col + e < a.N ? v8[e] : (half_t)-__builtin_huge_valf();
              uint32_t m = pk_max(m8);
              m = pk_max(m, (uint32_t)__shfl_xor((int)m, 1, 64), m);
              m = pk_max(m, (uint32_t)__shfl_xor((int)m, 2, 64), m);
              if (row < a.M && (sch & 3) == 0) a.bmax[(int64_t)row * a.ldb + col / LOGIT_BLOCK] = pk_larger(m);
            }
            if (row < a.M) {
              // uniform part + per-lane part computed once per tile: no per-strip vector multiply
              half_t* dst = a.out + ((int64_t)(m0 + wm * C::TM + fm * 32 + 8 * q) * a.ldo + n0 + wn * C::TN) + lane_off[p];
              if (!EDGE || col + 8 <= a.n_store) {
                if (!LOSS && a.through) store<THROUGH>(reinterpret_cast<half8*>(dst), v8);
                else store<PAST>(reinterpret_cast<half8*>(dst), v8);  // G is not re-read before it leaves the L2
              } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                  if (col + e < a.n_store) dst[e] = v8[e];
              }
            }
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
      }
    };
    if (n0 + C::BN > a.N || (LOSS && m0 + C::BM > a.M)) body(std::true_type{});
    else body(std::false_type{});
  };
  C::run(0, n_items, lds, get, epilogue);
  if constexpr (LOSS) {
    // deterministic: lanes -> wave (butterfly), waves -> workgroup (LDS, fixed order), one partial per workgroup
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss_acc += __shfl_xor(loss_acc, off, 64);
    double* red = reinterpret_cast<double*>(smem_raw);
    __syncthreads();
    if (lane == 0) red[wave] = loss_acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int i = 0; i < C::NW; ++i) t += red[i];
      a.loss_part[w] = t;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// positives: G -= 1 at the (row, label) pairs of a sparse label list, after the forward pass
// ---------------------------------------------------------------------------------------------
// One wave per pair.  The pair's logit is computed again, in fp32 from the fp16 operands (two rows of d, from the L2 or
// HBM), because G holds sigmoid(z) already rounded to fp16 and sigmoid(z) - 1 has to be rounded once, as a whole.  Pairs
// are independent: no pass over the list that sorts them by tile, no list look-up in the forward epilogue, and a pair
// listed twice writes the same value twice.  Input is CSR (rowptr/colidx, pos_x == nullptr; a pair finds its row by a
// 64-way search of the row pointers, two rounds of loads up to 4096 rows) or COO (pos_x/pos_y int64).  Pairs whose row
// or column is out of range are dropped.  (The pass that bucketed the list by label tile ran in one workgroup in front
// of the forward pass: 11.6 us at 2729 pairs, 23 us at 8357; this one takes 5.9 and 7.3, with the loss 8.0 at 2729.)
// LOSS: loss_pos[p] = z of the pair, or 0 if it was dropped or another copy of it was first.  The copies are told apart
// by G's sign bit, which sigmoid leaves clear and a visited positive sets (a zero difference is stored as -0).  This z is
// the forward pass's to the last bit, made by the same MFMAs in the same order: it cancels the max(z, 0) that the pass
// added, and a difference of 1e-6 between two sums of the same products is not small beside what is left, 4.5e-5 at z = 10.
enum PosMode { POS_G = 0, POS_LOSS_WIDE = 1, POS_LOSS = 2 };  // the loss with the z of fwd_wide_kernel or of fwd_kernel

template <int MODE>
__global__ void __launch_bounds__(256) positives_kernel(const half_t* __restrict__ X, int64_t ldx, const half_t* __restrict__ W,
                                                        int64_t ldw, const int32_t* __restrict__ rowptr,
                                                        const int32_t* __restrict__ colidx, const int64_t* __restrict__ pos_x,
                                                        const int64_t* __restrict__ pos_y, int64_t nnz, int B, int64_t L, int d,
                                                        half_t* G, int64_t ldg, float* __restrict__ loss_pos) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int KQ = MODE == POS_LOSS_WIDE ? 4 : 2;  // pieces of 8 k per MFMA
  [[maybe_unused]] __shared__ half8 xw_all[MODE == POS_G ? 1 : 4][2][64];
  [[maybe_unused]] half8 (&xw)[2][64] = xw_all[MODE == POS_G ? 0 : threadIdx.x >> 6];
  for (int64_t p = wave; p < nnz; p += (int64_t)gridDim.x * 4) {
    int64_t r = -1, c = -1;
    if (pos_x) {
      r = pos_x[p];
      c = pos_y[p];
    } else if (p >= rowptr[0] && p < rowptr[B]) {  // whatever the row pointers hold, an entry is read at most once
      c = colidx[p];
      int lo = 0, n = B;  // the row is the first b in [lo, lo + n) with rowptr[b + 1] > p
      while (n > 1) {
        const int step = (n + 63) >> 6, at = lo + min((lane + 1) * step, n);
        const unsigned long long above = __ballot(rowptr[at] > p);
        const int s = above ? __builtin_ctzll(above) : 63;
        lo += min(s * step, n - 1);
        n = min(step, B - lo);
        if (step == 1) break;
      }
      r = lo;
    }
    const bool in = r >= 0 && r < B && c >= 0 && c < L;
    float z = 0.f;
    [[maybe_unused]] std::conditional_t<MODE == POS_LOSS_WIDE, float4v, float16v> zc = {};
    if (in) {
      const half_t* x = X + r * ldx;
      const half_t* w = W + c * ldw;
      for (int k0 = 0; k0 < d; k0 += 512) {
        const int k = k0 + lane * 8;
        half8 xv = {}, wv = {};
        if (k < d) {
          xv = *reinterpret_cast<const half8*>(x + k);
          wv = *reinterpret_cast<const half8*>(w + k);
#pragma unroll
          for (int e = 0; e < 8; ++e) z = fmaf((float)xv[e], (float)wv[e], z);
        }
        if constexpr (MODE != POS_G) {
          // from "a lane has its eight k" to "a lane has those of its fragment" (zeros past d add nothing)
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          xw[0][lane] = xv;
          xw[1][lane] = wv;
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
          for (int q = 0; q < 64; q += KQ) {
            const half8 xf = xw[0][q + lane * KQ / 64], wf = xw[1][q + lane * KQ / 64];
            if constexpr (MODE == POS_LOSS_WIDE) zc = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, xf, zc, 0, 0, 0);
            else zc = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf, wf, zc, 0, 0, 0);
          }
          __builtin_amdgcn_wave_barrier();
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) z += __shfl_xor(z, off, 64);
      const half_t v = (half_t)(sigmoidf_fast(z) - 1.0f);
      if constexpr (MODE != POS_G) z = zc[0];  // every element of the block is the pair's z
      if (lane == 0) {
        half_t* g = G + r * ldg + c;
        if constexpr (MODE == POS_G) {
          *g = v;
        } else {
          const uint32_t bits = __builtin_bit_cast(uint16_t, v) | 0x8000u;
          const bool high = reinterpret_cast<uintptr_t>(g) & 2;
          uint32_t* word = reinterpret_cast<uint32_t*>(reinterpret_cast<uintptr_t>(g) & ~(uintptr_t)3);
          uint32_t old = *word;
          for (;;) {
            if (old & (high ? 0x80000000u : 0x8000u)) { z = 0.f; break; }  // another copy was first
            const uint32_t now = high ? (old & 0xffffu) | (bits << 16) : (old & 0xffff0000u) | bits;
            const uint32_t seen = atomicCAS(word, old, now);
            if (seen == old) break;
            old = seen;
          }
        }
      }
    }
    if constexpr (MODE != POS_G) { if (lane == 0) loss_pos[p] = z; }
  }
}

// Sum of the per-workgroup loss partials less the positives' logits, in double, in index order.
__global__ void __launch_bounds__(1024) loss_reduce_kernel(const double* __restrict__ part, int n, const float* __restrict__ pos,
                                                           int64_t n_pos, float* __restrict__ out) {
  __shared__ double wave_sum[16];
  double t = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) t += part[i];
  for (int64_t i = threadIdx.x; i < n_pos; i += 1024) t -= (double)pos[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
  if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) t += wave_sum[w];
    *out = (float)t;
  }
}

// ---------------------------------------------------------------------------------------------
// top-K for 8 < K <= 8192: exact selection over rows of fp16 logits (one workgroup per row)
// ---------------------------------------------------------------------------------------------
constexpr int SEL_MAX_K = 8192;  // at most half the capacity of the larger sort buffer
constexpr int SEL_THREADS = 1024;
constexpr int SEL_BINS = 2048;  // histogram over the top 11 bits of the 16-bit key
// candidates that are sorted in LDS: 2048 for K <= 1024 (the reference's K = 100 lives here), 16384 (128 KB of
// LDS, one row per CU at a time) for K up to SEL_MAX_K
constexpr int SEL_CAP_SMALL = 2048, SEL_CAP_LARGE = 16384;
constexpr int SEL_SMALL_MAX_K = SEL_CAP_SMALL / 2;
// At least K blocks reach the bound that the maxima give, on random logits up to a quarter more: the list of them has room for
// twice SEL_SMALL_MAX_K in the place of the histogram and, at the end of the large buffer, for 8192.  (64 rows x 1,310,720 x 64,
// K = 2049: 403 -> 143 us against full passes over the rows, which a list of 2048 led to; K = 8192, where it would not do: 649 -> 630.)
constexpr int SEL_LIST_LARGE = 8192, SEL_BLOCKS_MAX_K = SEL_LIST_LARGE * 3 / 4;
constexpr int SEL_BLOCKS_MIN = 2048;  // rows with fewer blocks of logits are selected without their maxima
static_assert(2 * SEL_MAX_K <= SEL_CAP_LARGE, "ranks per row");

// fp16 bit pattern -> 16-bit key that orders like the value (-0 counts as +0).
__device__ __forceinline__ uint32_t sel_key(uint32_t h) {
  if (h == 0x8000u) h = 0u;
  return (h & 0x8000u) ? (~h & 0xffffu) : (h | 0x8000u);
}
__device__ __forceinline__ uint32_t sel_unkey(uint32_t k) { return (k & 0x8000u) ? (k & 0x7fffu) : (~k & 0xffffu); }

template <int SEL_CAP>
struct SelLds {
  int hist[SEL_BINS];
  unsigned long long cand[SEL_CAP];
  int wave_tot[SEL_THREADS / 64];
  int n_cand, bin, above, n_blocks;
};

// The K largest of each row of `logits` (rows x L, leading dimension ldl, a multiple of 8), ordered by
// (value descending, label ascending).  Pass 1 histograms the top 11 key bits and finds the bin that
// holds the K-th largest; when at most SEL_CAP elements lie in that bin or above, they are gathered and
// sorted.  Otherwise pass 2 histograms the bin's low 5 bits to get the exact K-th key; elements above it
// are gathered, and the elements equal to it are taken in label order until K are found.
// With sample_stride > 1 the histogram is first taken over every sample_stride-th 16 KB block of the row
// only: the K-th largest of a subset is never above the K-th largest of the row, so every element in that
// bin or above is still a superset of the answer, about K * sample_stride elements; if they fit the sort
// buffer the row has been read 1 + 1/sample_stride times instead of twice, and if not the full passes run.
// With the maxima of the row's blocks of LOGIT_BLOCK (n_blocks > 0) they are that subset: the histogram is theirs, and only
// blocks whose maximum reaches the bound are read at all, about K of them.  A block that holds a value that is no number has
// no maximum to go by (one with the sign set ranks last); a row with such a block, or with more blocks at the bound than there is
// room for, goes on with the sampled pass.  (512 rows x 1,310,720 logits, K = 100: 368 us with the sampled pass, 54 with the
// maxima; the forward pass that leaves them takes as long as without.)
template <int SEL_CAP>
__global__ void __launch_bounds__(SEL_THREADS) topk_select_kernel(const half_t* __restrict__ logits, int64_t ldl, int L,
                                                                   int64_t numy, int K, int sample_stride,
                                                                   const half_t* __restrict__ bmax, int64_t ldb, int n_blocks,
                                                                   float* __restrict__ out_v,
                                                                   int64_t* __restrict__ out_i) {
  extern __shared__ __attribute__((aligned(16))) unsigned char sel_raw[];
  SelLds<SEL_CAP>& S = *reinterpret_cast<SelLds<SEL_CAP>*>(sel_raw);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint16_t* row = reinterpret_cast<const uint16_t*>(logits) + (int64_t)blockIdx.x * ldl;
  auto for_each_block = [&](int block_stride, auto&& f) {
    for (int64_t i64 = tid * 8; i64 < L; i64 += (int64_t)SEL_THREADS * 8 * block_stride) {
      const int i = (int)i64;
      const uint4v q = *reinterpret_cast<const uint4v*>(row + i);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (i + e < L) f(sel_key((q[e >> 1] >> (16 * (e & 1))) & 0xffffu), i + e);
    }
  };
  auto for_each = [&](auto&& f) { for_each_block(1, f); };
  // f(key, index) for every element of the row whose key is at least kthr.  Almost none is, so two elements at a
  // time are first tested in packed 16-bit arithmetic: flipping the magnitude bits of a negative fp16 pattern gives
  // a signed 16-bit integer x = key - 32768 (except that -0 gives -1 where its key is that of +0, hence the
  // threshold one lower), and min(x, t - 1) != x exactly when x >= t.  Only a 16-byte piece with a hit goes through
  // the exact per-element test.  Two pieces per thread are in flight.
  auto for_each_from = [&](const uint16_t* row, int L, uint32_t kthr, auto&& f) {
    typedef short short2v __attribute__((ext_vector_type(2)));
    const int xq = (int)kthr - 32768 - 1;  // quick test: x >= xq
    const bool all = xq <= -32768;
    const uint32_t t2 = ((uint32_t)(xq - 1) & 0xffffu) * 0x10001u;
    const short2v tv = __builtin_bit_cast(short2v, t2);
    auto piece = [&](const uint4v& q, int i) {
      uint32_t changed = 0u;
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        const uint32_t pair = q[e2];  // (a bit cast straight from the element expression reads element 0)
        const short2v h = __builtin_bit_cast(short2v, pair);
        const short2v x = h ^ ((h >> (short2v)(15)) & (short2v)(0x7fff));
        const short2v m = __builtin_elementwise_min(x, tv);
        changed |= __builtin_bit_cast(uint32_t, m) ^ __builtin_bit_cast(uint32_t, x);
      }
      if (all || changed != 0u) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t key = sel_key((q[e >> 1] >> (16 * (e & 1))) & 0xffffu);
          if (i + e < L && key >= kthr) f(key, i + e);
        }
      }
    };
    constexpr int64_t STEP = (int64_t)SEL_THREADS * 8;
    for (int64_t i64 = tid * 8; i64 < L; i64 += 2 * STEP) {
      const int i = (int)i64;
      const bool second = i64 + STEP < L;
      const uint4v q0 = *reinterpret_cast<const uint4v*>(row + i);
      uint4v q1 = {0u, 0u, 0u, 0u};
      if (second) q1 = *reinterpret_cast<const uint4v*>(row + i + STEP);
      piece(q0, i);
      if (second) piece(q1, i + (int)STEP);
    }
  };
  auto push_below = [&](int room, uint32_t key, int idx) {
    const int slot = atomicAdd(&S.n_cand, 1);
    if (slot < room) S.cand[slot] = ((unsigned long long)(0xffffu - key) << 32) | (uint32_t)idx;
  };
  auto push = [&](uint32_t key, int idx) { push_below(SEL_CAP, key, idx); };
  // Finds, over hist[0..nb), the highest bin b with (count in bins above b) + base < K <= that + hist[b];
  // writes S.bin = b and S.above = base + count above b.  nb is a multiple of 64; executed by wave 0.
  auto find_bin = [&](int nb, int base) {
    if (wave == 0) {
      const int per = nb / 64;
      int p = 0;
      for (int j = 0; j < per; ++j) p += S.hist[lane * per + j];
      int suf = p;  // sum over lanes >= this one
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_down(suf, off, 64);
        if (lane + off < 64) suf += v;
      }
      const unsigned long long m = __ballot(base + suf >= K);
      const int owner = 63 - __builtin_clzll(m | 1ull);  // m != 0 because K <= L
      if (lane == owner) {
        int above = base + suf - p, b = lane * per + per - 1;
        for (; b > lane * per; --b) {
          if (above + S.hist[b] >= K) break;
          above += S.hist[b];
        }
        S.bin = b;
        S.above = above;
      }
    }
  };

  for (int b = tid; b < SEL_BINS; b += SEL_THREADS) S.hist[b] = 0;
  if (tid == 0) S.n_cand = 0;
  __syncthreads();
  bool done = false;
  auto reset = [&]() {
    for (int b = tid; b < SEL_BINS; b += SEL_THREADS) S.hist[b] = 0;
    if (tid == 0) S.n_cand = 0;
    __syncthreads();
  };
  if (n_blocks > 0) {  // the host only gives maxima of at least K blocks
    const uint16_t* maxima = reinterpret_cast<const uint16_t*>(bmax) + (int64_t)blockIdx.x * ldb;
    if (tid == 0) S.bin = 0;
    __syncthreads();
    auto count = [&](uint32_t h) {
      if ((h & 0x7fffu) > 0x7c00u) S.bin = -1;
      atomicAdd(&S.hist[sel_key(h) >> 5], 1);
    };
    if (n_blocks >= SEL_THREADS * 8) {
      for (int i = tid * 8; i < n_blocks; i += SEL_THREADS * 8) {
        const uint4v q = *reinterpret_cast<const uint4v*>(maxima + i);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (i + e < n_blocks) count((q[e >> 1] >> (16 * (e & 1))) & 0xffffu);
      }
    } else {
      for (int i = tid; i < n_blocks; i += SEL_THREADS) count(maxima[i]);
    }
    __syncthreads();
    const bool numbers = S.bin == 0;
    __syncthreads();
    if (numbers) {
      find_bin(SEL_BINS, 0);
      __syncthreads();
      const uint32_t kthr = (uint32_t)S.bin << 5;
      // the blocks that reach the bound, in a list, then their logits, four threads to a block
      constexpr bool LARGE = SEL_CAP > SEL_CAP_SMALL;
      constexpr int LIST = LARGE ? SEL_LIST_LARGE : SEL_BINS, ROOM = LARGE ? SEL_CAP - LIST / 2 : SEL_CAP;
      int* const list = LARGE ? reinterpret_cast<int*>(S.cand + ROOM) : S.hist;
      if (tid == 0) S.n_blocks = 0;
      __syncthreads();
      for_each_from(maxima, n_blocks, kthr, [&](uint32_t, int b) {
        const int slot = atomicAdd(&S.n_blocks, 1);
        if (slot < LIST) list[slot] = b;
      });
      __syncthreads();
      const int hits = S.n_blocks;
      for (int t = tid; t < hits * 4 && hits <= LIST; t += SEL_THREADS) {
        const int i = list[t >> 2] * LOGIT_BLOCK + (t & 3) * 8;
        if (i < L) {
          const uint4v q = *reinterpret_cast<const uint4v*>(row + i);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t key = sel_key((q[e >> 1] >> (16 * (e & 1))) & 0xffffu);
            if (i + e < L && key >= kthr) push_below(ROOM, key, i + e);
          }
        }
      }
      __syncthreads();
      done = hits <= LIST && S.n_cand <= ROOM;
      __syncthreads();
    }
    if (!done) reset();
  }
  if (!done && sample_stride > 1) {
    for_each_block(sample_stride, [&](uint32_t key, int) { atomicAdd(&S.hist[key >> 5], 1); });
    __syncthreads();
    find_bin(SEL_BINS, 0);  // the host only asks for a sample that holds at least K elements
    __syncthreads();
    const int sbin = S.bin;
    for_each_from(row, L, (uint32_t)sbin << 5, [&](uint32_t key, int idx) { push(key, idx); });
    __syncthreads();
    done = S.n_cand <= SEL_CAP;  // counts every push, also those that found the buffer full
    __syncthreads();
    if (!done) reset();
  }
  int bin = 0, above = 0, in_bin = 0;
  if (!done) {
    for_each([&](uint32_t key, int) { atomicAdd(&S.hist[key >> 5], 1); });
    __syncthreads();
    find_bin(SEL_BINS, 0);
    __syncthreads();
    bin = S.bin;
    above = S.above;
    in_bin = S.hist[bin];
    __syncthreads();
  }
  if (done) {
    // the sampled bound already gathered a superset of the answer
  } else if (above + in_bin <= SEL_CAP) {
    for_each_from(row, L, (uint32_t)bin << 5, [&](uint32_t key, int idx) { push(key, idx); });
  } else {
    if (tid < 64) S.hist[tid] = 0;
    __syncthreads();
    for_each([&](uint32_t key, int) { if ((int)(key >> 5) == bin) atomicAdd(&S.hist[key & 31u], 1); });
    __syncthreads();
    find_bin(64, above);
    __syncthreads();
    const uint32_t thr = ((uint32_t)bin << 5) | (uint32_t)S.bin;
    const int n_gt = S.above, n_eq = S.hist[S.bin];
    __syncthreads();
    if (n_gt + n_eq <= SEL_CAP) {
      for_each_from(row, L, thr, [&](uint32_t key, int idx) { push(key, idx); });
    } else {
      // too many copies of the K-th value to sort: those above it first, then its copies in label order
      for_each_from(row, L, thr + 1u, [&](uint32_t key, int idx) { push(key, idx); });
      const int need = K - n_gt;
      int taken = 0;
      for (int base = 0; base < L && taken < need; base += SEL_THREADS * 8) {
        const int i = base + tid * 8;
        uint32_t hit = 0;
        if (i < L) {
          const uint4v q = *reinterpret_cast<const uint4v*>(row + i);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (i + e < L && sel_key((q[e >> 1] >> (16 * (e & 1))) & 0xffffu) == thr) hit |= 1u << e;
        }
        const int c = __builtin_popcount(hit);
        int inc = c;  // inclusive scan over the wave
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int v = __shfl_up(inc, off, 64);
          if (lane >= off) inc += v;
        }
        if (lane == 63) S.wave_tot[wave] = inc;
        __syncthreads();
        int before = 0, total = 0;
        for (int w = 0; w < SEL_THREADS / 64; ++w) {
          const int t = S.wave_tot[w];
          if (w < wave) before += t;
          total += t;
        }
        int rank = taken + before + inc - c;
        for (int e = 0; e < 8; ++e)
          if (hit & (1u << e)) {
            if (rank < need) S.cand[n_gt + rank] = ((unsigned long long)(0xffffu - thr) << 32) | (uint32_t)(i + e);
            ++rank;
          }
        taken += total;
        __syncthreads();
      }
      if (tid == 0) S.n_cand = K;
    }
  }
  __syncthreads();
  int fewest = 512;  // what would be sorted with a closer bound, a power of two that holds little more than K
  while (fewest < K + K / 16) fewest <<= 1;
  if (done && S.n_cand > (K < 128 ? 4 * K : fewest)) {
    // a loose bound: the K-th largest candidate's bin gives a closer one, and fewer to sort
    unsigned long long mine[SEL_CAP / SEL_THREADS];
    const int had = S.n_cand;
    for (int b = tid; b < SEL_BINS; b += SEL_THREADS) S.hist[b] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SEL_CAP / SEL_THREADS; ++j) {
      const int c = tid + j * SEL_THREADS;
      mine[j] = c < had ? S.cand[c] : ~0ull;
      if (c < had) atomicAdd(&S.hist[(0xffffu - (uint32_t)(mine[j] >> 32)) >> 5], 1);
    }
    __syncthreads();
    find_bin(SEL_BINS, 0);
    if (tid == 0) S.n_cand = 0;
    __syncthreads();
    const uint32_t kthr = (uint32_t)S.bin << 5;
#pragma unroll
    for (int j = 0; j < SEL_CAP / SEL_THREADS; ++j)
      if (tid + j * SEL_THREADS < had && 0xffffu - (uint32_t)(mine[j] >> 32) >= kthr) S.cand[atomicAdd(&S.n_cand, 1)] = mine[j];
    __syncthreads();
  }
  const int n = S.n_cand;  // K <= n <= SEL_CAP
  int n2 = 1;
  while (n2 < n) n2 <<= 1;
  for (int i = n + tid; i < n2; i += SEL_THREADS) S.cand[i] = ~0ull;
  __syncthreads();
  for (int k = 2; k <= n2; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = tid; i < n2; i += SEL_THREADS) {
        const int x = i ^ j;
        if (x > i) {
          const unsigned long long a = S.cand[i], b = S.cand[x];
          const bool up = (i & k) == 0;
          if ((a > b) == up) { S.cand[i] = b; S.cand[x] = a; }
        }
      }
      __syncthreads();
    }
  for (int r = tid; r < K; r += SEL_THREADS) {
    const unsigned long long c = S.cand[r];
    const uint32_t hbits = sel_unkey(0xffffu - (uint32_t)(c >> 32));
    const uint16_t h16 = (uint16_t)hbits;
    half_t h;
    __builtin_memcpy(&h, &h16, 2);
    int64_t idx = (int64_t)(uint32_t)c;
    if (idx >= numy) idx = numy - 1;
    out_v[(int64_t)blockIdx.x * K + r] = (float)h;
    out_i[(int64_t)blockIdx.x * K + r] = idx;
  }
}

// ---------------------------------------------------------------------------------------------
// dX = alpha * G . W (+ beta * dX): split over the label axis, fp32 partials, then a reduce
// ---------------------------------------------------------------------------------------------
// Batches above 128 rows: 256 dims (the A side, contiguous in dX) x 256 rows x 64 labels per stage.  W runs ahead.
using DxWide = WideCore<256, 256, 2, 2, false>;
using DxCore = PipeCore<128, 256, 64, 2, 4, 3, true, false, true, false, false, 4>;   // up to 128 rows; accumulators in AGPRs
using DxCore64 = PipeCore<64, 256, 64, 2, 4, 3, true, false, true, false, false, 4>;  // up to 64

struct DxArgs {
  const half_t* G; int64_t ldg;   // M x K, K-contiguous (K = labels)
  const half_t* W; int64_t ldw;   // K x N, N-contiguous
  float* part;                    // [splits][M][N]
  int M, N, K;
  int tiles_m, tiles_n, splits, k_per_split;  // k_per_split is a multiple of BK
};

// One workgroup per (output tile, slice of the label axis); the tiles of one slice get ids on one XCD.
template <int HOW>
__global__ void __launch_bounds__(DxWide::NT) dx_wide_kernel(DxArgs a) {
  using C = DxWide;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* lds = reinterpret_cast<half_t*>(smem_raw);
  int tile, split;
  xcd_map(blockIdx.x, a.tiles_m * a.tiles_n, tile, split);
  const int mt = tile % a.tiles_m, nt = tile / a.tiles_m;
  const int m0 = mt * C::BN, n0 = nt * C::BM;
  const int64_t kb64 = (int64_t)split * a.k_per_split;
  const int k_begin = (int)(kb64 < a.K ? kb64 : a.K);
  const int k_end = (int)(kb64 + a.k_per_split < a.K ? kb64 + a.k_per_split : a.K);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be
  const int wm = wave / C::WN, wn = wave % C::WN;
  float* part = a.part + (int64_t)split * a.M * a.N;
  auto leave = [&](float4v (&acc)[C::FM][C::FN]) {
#pragma unroll
    for (int fn = 0; fn < C::FN; ++fn) {
      const int row = m0 + wn * C::TN + fn * 16 + (lane & 15);
      if (row < a.M) {
#pragma unroll
        for (int fm = 0; fm < C::FM; ++fm) {
          const int col = n0 + wm * C::TM + fm * 16 + 4 * (lane >> 4);
          if (col < a.N) store<HOW>(reinterpret_cast<float4v*>(part + (int64_t)row * a.N + col), acc[fm][fn]);
        }
      }
    }
  };
  if (k_end <= k_begin) {  // a slice past the end of the label axis contributes zeros
    float4v acc[C::FM][C::FN];
    C::zero(acc);
    leave(acc);
    return;
  }
  auto get = [&](int, C::Operand& oa, C::Operand& ob, int& kb, int& ke) {
    oa = C::Operand{a.W, a.ldw, n0, a.N};
    ob = C::Operand{a.G, a.ldg, m0, a.M};
    kb = k_begin;
    ke = k_end;
  };
  auto epilogue = [&](int, float4v (&acc)[C::FM][C::FN]) { leave(acc); };
  C::run(0, 1, lds, get, epilogue);
}

// The same on the smaller row tiles.
template <class C, int HOW>
__global__ void __launch_bounds__(C::NT) dx_kernel(DxArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* lds = reinterpret_cast<half_t*>(smem_raw);
  int tile, split;
  xcd_map(blockIdx.x, a.tiles_m * a.tiles_n, tile, split);
  const int mt = tile % a.tiles_m, nt = tile / a.tiles_m;
  const int m0 = mt * C::BM, n0 = nt * C::BN;
  const int64_t kb64 = (int64_t)split * a.k_per_split;
  const int k_begin = (int)(kb64 < a.K ? kb64 : a.K);
  const int k_end = (int)(kb64 + a.k_per_split < a.K ? kb64 + a.k_per_split : a.K);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be
  const int wm = wave / C::WN, wn = wave % C::WN;
  float* part = a.part + (int64_t)split * a.M * a.N;
  auto leave = [&](float16v (&acc)[C::FM][C::FN]) {
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < C::FN; ++fn) {
        const int col = n0 + wn * C::TN + fn * 32 + (lane & 31);
        if (col < a.N) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = m0 + wm * C::TM + fm * 32 + c_row(r, lane);
            if (row < a.M) store<HOW>(part + (int64_t)row * a.N + col, (float)acc[fm][fn][r]);
          }
        }
      }
  };
  if (k_end <= k_begin) {  // a slice past the end of the label axis contributes zeros
    float16v acc[C::FM][C::FN];
    C::zero(acc);
    leave(acc);
    return;
  }
  auto get = [&](int, typename C::Operand& oa, typename C::Operand& ob, int& kb, int& ke) {
    oa = typename C::Operand{a.G, a.ldg, m0, a.M, a.K};
    ob = typename C::Operand{a.W, a.ldw, n0, a.N, a.K};
    kb = k_begin;
    ke = k_end;
  };
  auto epilogue = [&](int, float16v (&acc)[C::FM][C::FN]) { leave(acc); };
  C::run(0, 1, lds, get, epilogue);
}

// out[m][n] = alpha * sum_s part[s][m][n] + beta * out[m][n].  32 pieces of 4 columns per workgroup, SG threads to a piece,
// each taking every SG-th slice.  Bound by the latency of a thread's chain of loads when the output is small: one thread per
// piece walked all 256 slices of a small batch in 6 workgroups a CU or fewer (25.8 us at 32 x 768 x 256 slices, 36.7 at
// 256 x 384 x 256, 15.7 at 512 x 768 x 40; now 5.0, 11.5 and 11.4).
template <int SG>
__global__ void __launch_bounds__(32 * SG) dx_reduce_kernel(const float* __restrict__ part, float* __restrict__ out,
                                                            int64_t ldo, int M, int N, int splits, float alpha,
                                                            float beta) {
  __shared__ float4v red[SG / 2][32];
  const int piece = threadIdx.x & 31, sg = threadIdx.x >> 5;
  const int nq = N / 4;
  const int64_t q = (int64_t)blockIdx.x * 32 + piece;
  const bool in = q < (int64_t)M * nq;
  float4v s = {0.f, 0.f, 0.f, 0.f};
  if (in) {
    const float* p = part + q * 4;
#pragma unroll 8
    for (int i = sg; i < splits; i += SG) s += *reinterpret_cast<const float4v*>(p + (int64_t)i * M * N);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) s[e] += __shfl_xor(s[e], 32, 64);
  if (!(sg & 1)) red[sg >> 1][piece] = s;
  __syncthreads();
  if (sg != 0 || !in) return;
#pragma unroll
  for (int i = 1; i < SG / 2; ++i) s += red[i][piece];
  float* o = out + (q / nq) * ldo + (q % nq) * 4;
  float4v r = alpha * s;
  if (beta != 0.f) {
    r[0] += beta * o[0]; r[1] += beta * o[1]; r[2] += beta * o[2]; r[3] += beta * o[3];
  }
  o[0] = r[0]; o[1] = r[1]; o[2] = r[2]; o[3] = r[3];
}

// ---------------------------------------------------------------------------------------------
// dW = G^T . X; either written out (fp32, alpha/beta) or consumed by the momentum update
// ---------------------------------------------------------------------------------------------
// 256 labels x 256 dims x 64 batch rows per stage, eight waves of 64 labels x 128 dims, one workgroup per CU.
// (A 128 x 256 x 32 tile with four waves and two workgroups per CU measured 7-11 % slower at every batch size tried: its stages are half as
// deep, and move half again as much through LDS and the fetch path per flop.  DwCore128 keeps the depth of 64 rows and eight waves; per flop it
// moves twice what DwCore does, and is taken where that is not what binds.)
using DwCore = PipeCore<256, 256, 64, 4, 2, 2, false, false, false, false, false, 4>;
// 128 labels x 128 dims, eight waves of 32 x 64, two workgroups to a CU: see dw_plan.
using DwCore128 = PipeCore<128, 128, 64, 4, 2, 2, false, false, false, false, false, 4>;
static_assert(DwCore::BM == DW_TILE && DwCore::BN == DW_TILE && DwCore128::BM == DW_SMALL_TILE && DwCore128::BN == DW_SMALL_TILE, "tile_plan.hpp");
constexpr int DW_STAGE_FLOATS = 8 * 64;  // per wave: 8 label rows x 64 dims
template <class C>
struct DwLds {
  static constexpr int BYTES = C::LDS_BYTES + C::NW * DW_STAGE_FLOATS * 4, PER_CU = 160 * 1024 / BYTES;
  static_assert(BYTES <= 160 * 1024, "LDS budget");
  static_assert(C::FN % 2 == 0, "epilogue walks pairs of 32-column blocks");
};
static_assert(DwLds<DwCore>::PER_CU == 1 && DwLds<DwCore128>::PER_CU == 2, "workgroups on a CU");

struct DwArgs {
  const half_t* G; int64_t ldg;   // K x M (batch rows x labels), label-contiguous
  const half_t* X; int64_t ldx;   // K x N, N-contiguous
  int M, N, K;                    // labels, feature dims, batch rows
  int g_cols;                     // readable columns of G per row (>= M, multiple of 8)
  // DW_OUT
  float* out; int64_t ldo; float alpha, beta;
  // DW_UPDATE
  half_t* Wt; int64_t ldw; half_t* Mo; int64_t ldm; float lr, mu, wd;
  // DW_UPDATE_MASTER: fp32 master weights and momentum; Wt above receives the fp16 copy of the new weights
  float* W32; int64_t ldw32; float* M32; int64_t ldm32;
  float* dw_dump; int64_t ld_dump;  // optional copy of dW (may be null)
  int tiles_m, tiles_n, n_ids;      // n_ids = tiles_n * round_up(tiles_m, 8)
};

// Persistent, as many workgroups as the CUs hold: workgroup w takes tile ids w, w + gridDim.x, ...; the dim tiles of
// one label tile have neighbouring ids on one XCD, so its slice of G is fetched from HBM once.
// HOW what is written is stored: see dw_plan.
template <class C, int MODE, int HOW>
__global__ void __launch_bounds__(C::NT, C::NW * DwLds<C>::PER_CU / 4) dw_kernel(DwArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* lds = reinterpret_cast<half_t*>(smem_raw);
  const int G = gridDim.x, w = blockIdx.x;
  const int n_items = (a.n_ids - w + G - 1) / G;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be
  const int wm = wave / C::WN, wn = wave % C::WN;
  float* stage = reinterpret_cast<float*>(smem_raw + C::LDS_BYTES) + wave * DW_STAGE_FLOATS;

  auto get = [&](int item, typename C::Operand& oa, typename C::Operand& ob, int& kb, int& ke) {
    int nt, mt;
    xcd_map(item * G + w, a.tiles_n, nt, mt);
    oa = typename C::Operand{a.G, a.ldg, mt < a.tiles_m ? mt * C::BM : 0, a.g_cols, a.K};
    ob = typename C::Operand{a.X, a.ldx, nt * C::BN, a.N, a.K};
    kb = 0;
    ke = a.K;
  };
  auto epilogue = [&](int item, float16v (&acc)[C::FM][C::FN]) {
    int nt, mt;
    xcd_map(item * G + w, a.tiles_n, nt, mt);
    if (mt >= a.tiles_m) return;
    const int m0 = mt * C::BM, n0 = nt * C::BN;
    const int h = lane >> 5;
    const int srow = lane >> 3, sch = lane & 7;  // staging read: 8 rows x 8 chunks of 8 dims
    // The tile is walked in NS strips of 8 label rows x 64 dims per wave.  In DW_UPDATE mode the strip's
    // W and M pieces are fetched DEPTH strips ahead: one strip in flight per wave leaves HBM latency-bound.
    // They are read once per step, hence non-temporal (measured: 3 % off the kernel).
    constexpr int NS = C::FM * 4 * (C::FN / 2);
    constexpr int DEPTH = MODE == DW_UPDATE_MASTER ? 2 : 4;  // the fp32 pieces take twice the registers per strip (2-6 measure alike)
    auto strip_row = [&](int s) { return m0 + wm * C::TM + (s / (4 * (C::FN / 2))) * 32 + 8 * ((s / (C::FN / 2)) % 4) + srow; };
    auto strip_col = [&](int s) { return n0 + wn * C::TN + (s % (C::FN / 2)) * 64 + sch * 8; };
    // The fp32 arrays (dW out, master W and M) are touched in two 16-byte pieces per lane and strip.  With a lane
    // on 8 consecutive dims each piece's instruction would write every other 16 bytes of a line; there a lane
    // takes dims c .. c+3 and c+32 .. c+35 instead, so that eight lanes cover a whole 128-byte line each time.
    constexpr bool SPLIT = MODE != DW_UPDATE;
    auto split_col = [&](int s) { return n0 + wn * C::TN + (s % (C::FN / 2)) * 64 + sch * 4; };
    half8 wq[DEPTH], mq[DEPTH];
    float4v w32q[DEPTH][2], m32q[DEPTH][2];  // DW_UPDATE_MASTER
    auto fetch32 = [&](int s, float4v (&wv)[2], float4v (&mv)[2]) {
      int row = strip_row(s), c0 = split_col(s), c1 = c0 + 32;
      row = row < a.M ? row : a.M - 1;
      c0 = c0 < a.N ? c0 : a.N - 4;
      c1 = c1 < a.N ? c1 : a.N - 4;
      const float* wp = a.W32 + (int64_t)row * a.ldw32;
      const float* mp = a.M32 + (int64_t)row * a.ldm32;
      wv[0] = __builtin_nontemporal_load(reinterpret_cast<const float4v*>(wp + c0));
      wv[1] = __builtin_nontemporal_load(reinterpret_cast<const float4v*>(wp + c1));
      mv[0] = __builtin_nontemporal_load(reinterpret_cast<const float4v*>(mp + c0));
      mv[1] = __builtin_nontemporal_load(reinterpret_cast<const float4v*>(mp + c1));
    };
    // unconditional (out-of-range strips read the last valid row / column block and are not stored):
    // straight-line loads let the compiler count exactly how many may stay in flight at each use
    auto fetch = [&](int s, half8& wv, half8& mv) {
      int row = strip_row(s), col = strip_col(s);
      row = row < a.M ? row : a.M - 1;
      col = col < a.N ? col : a.N - 8;
      wv = __builtin_nontemporal_load(reinterpret_cast<const half8*>(a.Wt + (int64_t)row * a.ldw + col));
      mv = __builtin_nontemporal_load(reinterpret_cast<const half8*>(a.Mo + (int64_t)row * a.ldm + col));
    };
    if constexpr (MODE == DW_UPDATE) {
#pragma unroll
      for (int s = 0; s < DEPTH && s < NS; ++s) fetch(s, wq[s], mq[s]);
    }
    if constexpr (MODE == DW_UPDATE_MASTER) {
#pragma unroll
      for (int s = 0; s < DEPTH && s < NS; ++s) fetch32(s, w32q[s], m32q[s]);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int fm = s / (4 * (C::FN / 2)), q = (s / (C::FN / 2)) % 4, fp = s % (C::FN / 2);
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          stage[(4 * h + rr) * 64 + f * 32 + (lane & 31)] = acc[fm][2 * fp + f][4 * q + rr];
      // the wave's own LDS traffic is ordered: the writes above are visible to the reads below
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      const float4v v0 = *reinterpret_cast<const float4v*>(stage + srow * 64 + (SPLIT ? sch * 4 : sch * 8));
      const float4v v1 = *reinterpret_cast<const float4v*>(stage + srow * 64 + (SPLIT ? 32 + sch * 4 : sch * 8 + 4));
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int row = strip_row(s), col = SPLIT ? split_col(s) : strip_col(s);
      const int col1 = SPLIT ? col + 32 : col + 4;  // first dim of the lane's second piece
      const bool in = row < a.M && col < a.N, in1 = row < a.M && col1 < a.N;
      const float g[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
      if constexpr (MODE == DW_OUT) {
        float* orow = a.out + (int64_t)row * a.ldo;
        float4v o0, o1;
#pragma unroll
        for (int e = 0; e < 4; ++e) { o0[e] = a.alpha * g[e]; o1[e] = a.alpha * g[4 + e]; }
        if (a.beta != 0.f) {  // both pieces' loads before either store
          float4v p0 = {0.f, 0.f, 0.f, 0.f}, p1 = {0.f, 0.f, 0.f, 0.f};
          if (in) p0 = *reinterpret_cast<const float4v*>(orow + col);
          if (in1) p1 = *reinterpret_cast<const float4v*>(orow + col1);
          o0 += a.beta * p0;
          o1 += a.beta * p1;
        }
        if (in) store<HOW>(reinterpret_cast<float4v*>(orow + col), o0);
        if (in1) store<HOW>(reinterpret_cast<float4v*>(orow + col1), o1);
      } else if constexpr (MODE == DW_UPDATE_MASTER) {
        // the reference's regime (fp32 parameter and FusedSGD state, dl_base.py:185, main.py:178-179) with the
        // per-step fp16 cast of W (dl_base.py:562) written from the same pass
        float4v wv[2] = {w32q[s % DEPTH][0], w32q[s % DEPTH][1]}, mv[2] = {m32q[s % DEPTH][0], m32q[s % DEPTH][1]};
        if (s + DEPTH < NS) fetch32(s + DEPTH, w32q[s % DEPTH], m32q[s % DEPTH]);
        if (in) {  // the second piece lies 32 dims past the first: when it is inside N, so is the first
          if (a.dw_dump) {
            float* d = a.dw_dump + (int64_t)row * a.ld_dump;
            *reinterpret_cast<float4v*>(d + col) = v0;
            if (in1) *reinterpret_cast<float4v*>(d + col1) = v1;
          }
          half8 w16;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float wf = wv[e >> 2][e & 3];
            const float gg = g[e] + a.wd * wf;
            const float mf = a.mu * mv[e >> 2][e & 3] + gg;
            float wn = wf - a.lr * mf;
            // the copy is the rounding of the stored fp32 weight, as the reference's cast is (dl_base.py:562):
            // the empty statement keeps the compiler from fusing the subtraction and the conversion into one
            // mixed-precision instruction, which would round the exact difference to fp16 in one step
            asm volatile("" : "+v"(wn));
            mv[e >> 2][e & 3] = mf;
            wv[e >> 2][e & 3] = wn;
            w16[e] = (half_t)wn;
          }
          typedef _Float16 half4 __attribute__((ext_vector_type(4)));
          float* wp = a.W32 + (int64_t)row * a.ldw32;
          float* mp = a.M32 + (int64_t)row * a.ldm32;
          half_t* hp = a.Wt + (int64_t)row * a.ldw;
          store<HOW>(reinterpret_cast<float4v*>(mp + col), mv[0]);
          store<HOW>(reinterpret_cast<float4v*>(wp + col), wv[0]);
          store<HOW == THROUGH ? THROUGH : CACHED>(reinterpret_cast<half4*>(hp + col), half4{w16[0], w16[1], w16[2], w16[3]});
          if (in1) {
            store<HOW>(reinterpret_cast<float4v*>(mp + col1), mv[1]);
            store<HOW>(reinterpret_cast<float4v*>(wp + col1), wv[1]);
            store<HOW == THROUGH ? THROUGH : CACHED>(reinterpret_cast<half4*>(hp + col1), half4{w16[4], w16[5], w16[6], w16[7]});
          }
        }
      } else {
        half8 wv = wq[s % DEPTH], mv = mq[s % DEPTH];
        if (s + DEPTH < NS) fetch(s + DEPTH, wq[s % DEPTH], mq[s % DEPTH]);
        if (in) {
          if (a.dw_dump) {
            float* d = a.dw_dump + (int64_t)row * a.ld_dump + col;
            *reinterpret_cast<float4v*>(d) = v0;
            *reinterpret_cast<float4v*>(d + 4) = v1;
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float wf = (float)wv[e];
            const float gg = g[e] + a.wd * wf;
            const float mf = a.mu * (float)mv[e] + gg;
            mv[e] = (half_t)mf;
            wv[e] = (half_t)(wf - a.lr * mf);
          }
          store<HOW>(reinterpret_cast<half8*>(a.Mo + (int64_t)row * a.ldm + col), mv);
          store<HOW>(reinterpret_cast<half8*>(a.Wt + (int64_t)row * a.ldw + col), wv);
        }
      }
    }
  };
  C::run(0, n_items, lds, get, epilogue);
}

// ---------------------------------------------------------------------------------------------
// any-stride fallback: 64 x 64 output tile per workgroup, 4 x 4 outputs per thread, operands staged through LDS
// as fp32 in 32-deep slabs.  Each output is one fp32 accumulator summed over k in ascending order.  A slab is
// read with consecutive threads along whichever of its two axes has the smaller stride.
// ---------------------------------------------------------------------------------------------
constexpr int GEN_T = 64, GEN_K = 32, GEN_PAD = 4;
__global__ void __launch_bounds__(256) generic_gemm_kernel(const half_t* __restrict__ A, int64_t as0, int64_t as1,
                                                           const half_t* __restrict__ Bm, int64_t bs0, int64_t bs1,
                                                           void* out, int64_t os0, int64_t os1, int M, int N, int K,
                                                           float alpha, float beta, int sigmoid, int out_half) {
  __shared__ __align__(16) float As[GEN_K][GEN_T + GEN_PAD];
  __shared__ __align__(16) float Bs[GEN_K][GEN_T + GEN_PAD];
  const int tiles_n = (N + GEN_T - 1) / GEN_T;
  const int m0 = (int)(blockIdx.x / tiles_n) * GEN_T, n0 = (int)(blockIdx.x % tiles_n) * GEN_T;
  const int t = threadIdx.x, ty = t >> 4, tx = t & 15;
  const bool a_k_fast = (as1 < 0 ? -as1 : as1) <= (as0 < 0 ? -as0 : as0);
  const bool b_k_fast = (bs0 < 0 ? -bs0 : bs0) <= (bs1 < 0 ? -bs1 : bs1);
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += GEN_K) {
#pragma unroll
    for (int j = 0; j < GEN_T * GEN_K / 256; ++j) {
      const int i = t + j * 256;
      int kk = a_k_fast ? i % GEN_K : i / GEN_T, mm = a_k_fast ? i / GEN_K : i % GEN_T;
      As[kk][mm] = (m0 + mm < M && k0 + kk < K) ? (float)A[(int64_t)(m0 + mm) * as0 + (int64_t)(k0 + kk) * as1] : 0.f;
      kk = b_k_fast ? i % GEN_K : i / GEN_T;
      const int nn = b_k_fast ? i / GEN_K : i % GEN_T;
      Bs[kk][nn] = (n0 + nn < N && k0 + kk < K) ? (float)Bm[(int64_t)(k0 + kk) * bs0 + (int64_t)(n0 + nn) * bs1] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GEN_K; ++kk) {
      const float4 av = *reinterpret_cast<const float4*>(&As[kk][ty * 4]);
      const float4 bv = *reinterpret_cast<const float4*>(&Bs[kk][tx * 4]);
      const float a4[4] = {av.x, av.y, av.z, av.w}, b4[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += a4[i] * b4[j];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m >= M || n >= N) continue;
      float v = acc[i][j] * alpha;
      const int64_t o = (int64_t)m * os0 + (int64_t)n * os1;
      if (out_half) {
        half_t* p = reinterpret_cast<half_t*>(out) + o;
        if (beta != 0.f) v += beta * (float)*p;
        if (sigmoid) v = sigmoidf_fast(v);
        *p = (half_t)v;
      } else {
        float* p = reinterpret_cast<float*>(out) + o;
        if (beta != 0.f) v += beta * *p;
        if (sigmoid) v = sigmoidf_fast(v);
        *p = v;
      }
    }
}

// Plain copy, 16 bytes per thread step: the known-size kernel that HBM traffic counters are scaled by.
__global__ void __launch_bounds__(256) copy_kernel(const uint4v* __restrict__ src, uint4v* __restrict__ dst, int64_t n16) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

// SGD-momentum on an fp32 gradient (used when dW was accumulated over micro-batches).
__global__ void __launch_bounds__(256) sgd_momentum_kernel(half_t* __restrict__ W, half_t* __restrict__ Mo,
                                                           const float* __restrict__ grad, int64_t n8, float lr,
                                                           float mu, float wd) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  half8 w = reinterpret_cast<half8*>(W)[i];
  half8 m = reinterpret_cast<half8*>(Mo)[i];
  const float4v g0 = reinterpret_cast<const float4v*>(grad)[2 * i];
  const float4v g1 = reinterpret_cast<const float4v*>(grad)[2 * i + 1];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float wf = (float)w[e];
    const float gg = (e < 4 ? g0[e] : g1[e - 4]) + wd * wf;
    const float mf = mu * (float)m[e] + gg;
    m[e] = (half_t)mf;
    w[e] = (half_t)(wf - lr * mf);
  }
  reinterpret_cast<half8*>(W)[i] = w;
  reinterpret_cast<half8*>(Mo)[i] = m;
}

// The same on fp32 master weights and momentum, writing the fp16 copy of the new weights as well.
__global__ void __launch_bounds__(256) sgd_momentum_master_kernel(float* __restrict__ W32, float* __restrict__ M32,
                                                                  half_t* __restrict__ W16, const float* __restrict__ grad,
                                                                  int64_t n8, float lr, float mu, float wd) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  float4v w[2] = {reinterpret_cast<float4v*>(W32)[2 * i], reinterpret_cast<float4v*>(W32)[2 * i + 1]};
  float4v m[2] = {reinterpret_cast<float4v*>(M32)[2 * i], reinterpret_cast<float4v*>(M32)[2 * i + 1]};
  const float4v g[2] = {reinterpret_cast<const float4v*>(grad)[2 * i], reinterpret_cast<const float4v*>(grad)[2 * i + 1]};
  half8 h;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float wf = w[e >> 2][e & 3];
    const float mf = mu * m[e >> 2][e & 3] + g[e >> 2][e & 3] + wd * wf;
    float wn = wf - lr * mf;
    asm volatile("" : "+v"(wn));  // the copy is the rounding of the stored fp32 value (see dw_kernel)
    m[e >> 2][e & 3] = mf;
    w[e >> 2][e & 3] = wn;
    h[e] = (half_t)wn;
  }
  reinterpret_cast<float4v*>(W32)[2 * i] = w[0];
  reinterpret_cast<float4v*>(W32)[2 * i + 1] = w[1];
  reinterpret_cast<float4v*>(M32)[2 * i] = m[0];
  reinterpret_cast<float4v*>(M32)[2 * i + 1] = m[1];
  reinterpret_cast<half8*>(W16)[i] = h;
}

}  // namespace xfc

// Scratch of xfc_fwd_grad_csr_static: one copy per GPU, held until the process ends.  In host code the
// name is only a handle for hipGetSymbolAddress; kernels get the per-device address it returns.
static __device__ __align__(256) unsigned char g_static_scratch[XFC_STATIC_SCRATCH_BYTES];

// =============================================================================================
// C ABI
// =============================================================================================
using namespace xfc;

namespace {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_launch() {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    fprintf(stderr, "xfc: kernel launch failed: %s\n", hipGetErrorString(e));
    return XFC_ERR_HIP;
  }
  return XFC_OK;
}

constexpr int MAX_DEVICES = 64;
int current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) dev = 0;
  return dev;
}

constexpr int FULL_LDS = 160 * 1024;

// Dynamic LDS above the default limit needs the attribute once per kernel and device.
template <auto Kernel>
hipError_t raise_lds_limit(int lds) {
  static std::atomic<bool> raised[MAX_DEVICES];
  const int dev = current_device();
  if (lds <= 48 * 1024 || raised[dev].load(std::memory_order_acquire)) return hipSuccess;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e == hipSuccess) raised[dev].store(true, std::memory_order_release);
  return e;
}

// Launches Kernel and returns XFC_OK or XFC_ERR_HIP; nothing is launched when the LDS limit cannot be raised.
template <auto Kernel, class A>
int launch_k(dim3 g, dim3 b, int lds, hipStream_t st, const A& args) {
  const hipError_t e = raise_lds_limit<Kernel>(lds);
  if (e != hipSuccess) {
    fprintf(stderr, "xfc: cannot raise the dynamic LDS limit to %d bytes: %s\n", lds, hipGetErrorString(e));
    return XFC_ERR_HIP;
  }
  hipLaunchKernelGGL(Kernel, g, b, lds, st, args);
  return check_launch();
}

int num_cus() {
  static std::atomic<int> n[MAX_DEVICES];
  const int dev = current_device();
  int v = n[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int cnt = 0;
    if (hipDeviceGetAttribute(&cnt, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cnt <= 0) cnt = 256;
    v = cnt;
    n[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

// Device address of g_static_scratch on the current device (each GPU holds its own copy at its own
// address), looked up once per device; nullptr with the error printed if the lookup fails.
void* static_scratch_ptr() {
  static std::atomic<void*> ptr[MAX_DEVICES];
  const int dev = current_device();
  void* p = ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_static_scratch));
    if (e != hipSuccess || p == nullptr) {
      fprintf(stderr, "xfc: hipGetSymbolAddress(static scratch) failed: %s\n", hipGetErrorString(e));
      return nullptr;
    }
    ptr[dev].store(p, std::memory_order_release);
  }
  return p;
}

// Scratch of the forward pass with the loss: a double per forward workgroup and a float per label pair.
constexpr size_t LOSS_PART_BYTES = 4096;
size_t fwd_ws_bytes(int64_t nnz) { return LOSS_PART_BYTES + (size_t)round_up((nnz > 0 ? nnz : 1) * 4, 256); }

// Row-tile height for a batch of M rows (see FwdWide / FwdCore / FwdCore64).
inline int row_tile(int64_t M) { return M <= 64 ? 64 : M <= 128 ? 128 : 256; }

// Where the forward pass leaves the loss's partial sums, and how many: the workspace need not be aligned.
struct LossPart {
  double* at;
  int64_t places;
};
constexpr LossPart NO_LOSS = {nullptr, ANY_GRID};
LossPart loss_part_of(void* ws) {
  const uintptr_t from = (reinterpret_cast<uintptr_t>(ws) + 7) & ~(uintptr_t)7;
  return {reinterpret_cast<double*>(from), (int64_t)(reinterpret_cast<uintptr_t>(ws) + LOSS_PART_BYTES - from) / 64 * 8};
}

template <class C>
int launch_fwd_wide(int mode, const FwdArgs& a, dim3 g, hipStream_t st) {
  constexpr int LDS = C::LDS_BYTES;
  const dim3 b(C::NT);
  if (a.loss_part) return launch_k<fwd_wide_kernel<C, FWD_SIGMOID_PLAIN, false, true>>(g, b, LDS, st, a);
  if (mode == FWD_SIGMOID && a.beta != 0.f) return launch_k<fwd_wide_kernel<C, FWD_SIGMOID, true>>(g, b, LDS, st, a);
  if (mode == FWD_SIGMOID && a.alpha == 1.0f) return launch_k<fwd_wide_kernel<C, FWD_SIGMOID_PLAIN, false>>(g, b, LDS, st, a);
  if (mode == FWD_SIGMOID) return launch_k<fwd_wide_kernel<C, FWD_SIGMOID, false>>(g, b, LDS, st, a);
  if (a.bmax) return launch_k<fwd_wide_kernel<C, FWD_LINEAR, false, false, true>>(g, b, LDS, st, a);
  return launch_k<fwd_wide_kernel<C, FWD_LINEAR, false>>(g, b, LDS, st, a);
}

template <class C>
int launch_fwd_c(int mode, const FwdArgs& a, dim3 g, hipStream_t st) {
  constexpr int LDS = FwdLds<C>::BYTES;
  const dim3 b(C::NT);
  if (a.loss_part) return launch_k<fwd_kernel<C, FWD_SIGMOID_PLAIN, false, true>>(g, b, LDS, st, a);
  if (mode == FWD_SIGMOID && a.beta != 0.f) return launch_k<fwd_kernel<C, FWD_SIGMOID, true>>(g, b, LDS, st, a);
  if (mode == FWD_SIGMOID && a.alpha == 1.0f) return launch_k<fwd_kernel<C, FWD_SIGMOID_PLAIN, false>>(g, b, LDS, st, a);
  if (mode == FWD_SIGMOID) return launch_k<fwd_kernel<C, FWD_SIGMOID, false>>(g, b, LDS, st, a);
  if (a.bmax) return launch_k<fwd_kernel<C, FWD_LINEAR, false, false, true>>(g, b, LDS, st, a);
  return launch_k<fwd_kernel<C, FWD_LINEAR, false>>(g, b, LDS, st, a);
}

int launch_fwd(const FwdPlan& p, int mode, const half_t* X, int64_t ldx, const half_t* W, int64_t ldw, half_t* out, int64_t ldo, int M,
               int N, int K, int n_store, float alpha, float beta, hipStream_t st, LossPart loss = NO_LOSS,
               half_t* bmax = nullptr, int64_t ldb = 0) {
  FwdArgs a;
  a.X = X; a.ldx = ldx; a.W = W; a.ldw = ldw; a.out = out; a.ldo = ldo;
  a.M = M; a.N = p.first < N ? (int)p.first : N; a.K = K; a.n_store = (int)p.first; a.alpha = alpha; a.beta = beta;
  a.loss_part = loss.at; a.loss_have = 0;
  a.bmax = bmax; a.ldb = ldb;
  // Few logits are written through: with whole steps of 40 rows x 30,001 labels x 64 dims 23.0 -> 22.3 us, 256 x 20,001 x 256 43.2 -> 42.3, 50 x
  // 10,001 x 1024 41.4 -> 39.3, but (the wide loop's pieces are half lines) 512 x 20,001 x 768 97.2 -> 98.9, 100 x 60,001 109.9 -> 110.7.
  a.through = (int64_t)M * n_store * 2 <= (int64_t)(p.tile == FWD_WIDE128 ? 10 : 8) << 20;
  auto tiles = [&](FwdTile t, int64_t n) {
    a.tiles_n = ceil_div(n, fwd_tile_labels(t));
    const int64_t ids = fwd_ids(t, M, n);
    a.tiles_m = (int)(ids / round_up(a.tiles_n, 8));
    a.n_ids = (int)ids;
    return ids <= 0x7fffffff;
  };
  if (M <= 0 || n_store <= 0) return XFC_OK;
  if (!tiles(p.tile, p.first)) return XFC_ERR_INVALID;
  const int64_t grid = fwd_grid(p, M, num_cus(), loss.places), rest = fwd_rest_grid(p, M, n_store, num_cus(), loss.places);
  const dim3 g((unsigned)grid);
  int rc;
  switch (p.tile) {
    case FWD_64: rc = launch_fwd_c<FwdCore64>(mode, a, g, st); break;
    case FWD_128: rc = launch_fwd_c<FwdCore>(mode, a, g, st); break;
    case FWD_WIDE: rc = launch_fwd_wide<FwdWide>(mode, a, g, st); break;
    default: rc = launch_fwd_wide<FwdWide128>(mode, a, g, st); break;
  }
  if (rc || rest == 0) return rc;
  // the labels that whole rounds have left (a multiple of 256 lies before them)
  a.W += p.first * ldw;
  a.out += p.first;
  a.N = N - (int)p.first;
  a.n_store = n_store - (int)p.first;
  a.loss_have = (int)grid;
  if (bmax) a.bmax += p.first / LOGIT_BLOCK;
  tiles(FWD_WIDE128, a.n_store);
  return launch_fwd_wide<FwdWide128>(mode, a, dim3((unsigned)rest), st);
}

// Split count for dX: a multiple of 8 slices of the label axis (workgroup ids are dealt round-robin over
// the 8 XCDs, so the tiles of one slice then meet in one L2), each slice a multiple of the k-step.  The
// count minimises a cost model: workgroups run in rounds of one per CU, every workgroup pays a fixed prologue +
// partial-tile store, and the partial sums are written and read once.  A stage of a smaller row tile takes
// proportionally less time.  The model's constants were fitted to an eight-wave loop (2.4 us a stage; dx_wide_kernel takes
// 1.6) and a slower reduction; what decides is the number of rounds, which they do not touch.  Timed over 8 to 256 slices
// at 199, 256, 512 and 1024 rows x 131,072, 320,001 (384 dims), 655,363, 1,310,720 and 2,812,281 labels, the chosen count
// is within 1.6 % of the best one everywhere but at 199 x 131,072, where 64 slices take 67 us and the chosen 80 take 71
// to 74.
// With ws_limit the choice is restricted to slice counts whose partial sums fit that many bytes (8 slices, the
// minimum, is always a candidate: the caller checks the final need).  The unrestricted need is not monotone in M
// (a smaller batch may pick more slices), so a workspace sized for one batch serves smaller ones through this limit.
void dx_plan(int M, int N, int K, int& tiles_m, int& tiles_n, int& splits, int& k_per_split,
             size_t ws_limit = ~(size_t)0) {
  const int bm = row_tile(M);
  tiles_m = ceil_div(M, bm);
  tiles_n = ceil_div(N, DxWide::BM);
  const int64_t tiles = (int64_t)tiles_m * tiles_n > 0 ? (int64_t)tiles_m * tiles_n : 1;
  const int cus = num_cus();
  const double nk = (double)ceil_div(K, DxWide::BK);
  const int max_s = (int)round_up(ceil_div(K, DxWide::BK), 8);
  const double STAGE_US = 2.4 * (bm + 256) / 512.0;
  constexpr double FIXED_STAGES = 6.0, PART_BYTES_PER_US = 3.0e6;
  int best = 8;
  double best_cost = 0.0;
  for (int s = 8; s <= 256 && s <= max_s; s += 8) {
    if (s > 8 && (size_t)s * (size_t)M * (size_t)N * 4 > ws_limit) break;
    const double rounds = (double)ceil_div(tiles * s, cus);
    const double cost = rounds * (nk / s + FIXED_STAGES) * STAGE_US + 2.0 * s * (double)M * N * 4.0 / PART_BYTES_PER_US;
    if (s == 8 || cost < best_cost) { best = s; best_cost = cost; }
  }
  k_per_split = (int)round_up(ceil_div(K, best), DxWide::BK);
  splits = best;
}

void launch_dx_reduce(const float* part, float* out, int64_t ldo, int M, int N, int splits, float alpha, float beta,
                      hipStream_t st) {
  // threads to a piece: as many as keep the slices of a small output in flight at once; a large one fills the chip with 8
  const int64_t blocks = ceil_div((int64_t)M * (N / 4), 32);
  auto reduce = [&](auto kernel, int sg) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(32 * sg), 0, st, part, out, ldo, M, N, splits, alpha, beta);
  };
  if (blocks < 1024) reduce(dx_reduce_kernel<32>, 32);
  else reduce(dx_reduce_kernel<8>, 8);
}

int launch_dx(const half_t* G, int64_t ldg, const half_t* W, int64_t ldw, float* out, int64_t ldo, int M, int N, int K,
              float alpha, float beta, void* ws, size_t ws_bytes, hipStream_t st) {
  DxArgs a;
  dx_plan(M, N, K, a.tiles_m, a.tiles_n, a.splits, a.k_per_split, ws ? ws_bytes : 0);
  const size_t need = (size_t)a.splits * M * N * 4;
  if (ws == nullptr || ws_bytes < need) return XFC_ERR_WORKSPACE;
  a.G = G; a.ldg = ldg; a.W = W; a.ldw = ldw; a.part = reinterpret_cast<float*>(ws);
  a.M = M; a.N = N; a.K = K;
  const int64_t grid = (int64_t)a.tiles_m * a.tiles_n * a.splits;
  if (grid <= 0 || M <= 0 || N <= 0) return XFC_OK;
  const dim3 g((unsigned)grid);
  int rc;
  auto launch = [&](auto how) {
    constexpr int HOW = decltype(how)::value;
    switch (row_tile(M)) {
      case 64: return launch_k<dx_kernel<DxCore64, HOW>>(g, dim3(DxCore64::NT), DxCore64::LDS_BYTES, st, a);
      case 128: return launch_k<dx_kernel<DxCore, HOW>>(g, dim3(DxCore::NT), DxCore::LDS_BYTES, st, a);
      default: return launch_k<dx_wide_kernel<HOW>>(g, dim3(DxWide::NT), DxWide::LDS_BYTES, st, a);
    }
  };
  const bool through = dx_how(M, N, K, (int64_t)need, whole_lines(a.part, N, N, 4)) == THROUGH;
  rc = through ? launch(std::integral_constant<int, THROUGH>{}) : launch(std::integral_constant<int, CACHED>{});
  if (rc) return rc;
  launch_dx_reduce(a.part, out, ldo, M, N, a.splits, alpha, beta, st);
  return check_launch();
}

template <class C>
int launch_dw_tiles(DwMode mode, DwArgs a, StoreHow how, hipStream_t st) {
  a.tiles_m = ceil_div(a.M, C::BM);
  a.tiles_n = ceil_div(a.N, C::BN);
  const int64_t ids = (int64_t)a.tiles_n * round_up(a.tiles_m, 8);
  if (ids <= 0) return XFC_OK;
  if (ids > 0x7fffffff) return XFC_ERR_INVALID;
  a.n_ids = (int)ids;
  int64_t grid = (int64_t)DwLds<C>::PER_CU * round_up(num_cus(), 8);
  if (grid > ids) grid = ids / 8 * 8 > 0 ? ids / 8 * 8 : ids;
  const dim3 g((unsigned)grid), b(C::NT);
  constexpr int LDS = DwLds<C>::BYTES;
  auto launch = [&](auto mode_tag) {
    constexpr int MODE = decltype(mode_tag)::value;
    if (how == PAST) return launch_k<dw_kernel<C, MODE, PAST>>(g, b, LDS, st, a);
    if (how == THROUGH) return launch_k<dw_kernel<C, MODE, THROUGH>>(g, b, LDS, st, a);
    return launch_k<dw_kernel<C, MODE, CACHED>>(g, b, LDS, st, a);
  };
  if (mode == DW_UPDATE) return launch(std::integral_constant<int, DW_UPDATE>{});
  if (mode == DW_UPDATE_MASTER) return launch(std::integral_constant<int, DW_UPDATE_MASTER>{});
  return launch(std::integral_constant<int, DW_OUT>{});
}
int launch_dw(DwMode mode, const DwArgs& a, hipStream_t st) {
  const bool lines = mode == DW_OUT      ? whole_lines(a.out, a.ldo, a.N, 4)
                     : mode == DW_UPDATE ? whole_lines(a.Wt, a.ldw, a.N, 2) && whole_lines(a.Mo, a.ldm, a.N, 2)
                                         : whole_lines(a.W32, a.ldw32, a.N, 4) && whole_lines(a.M32, a.ldm32, a.N, 4);
  const DwPlan p = dw_plan(mode, a.M, a.N, a.K, lines, num_cus());
  return p.small ? launch_dw_tiles<DwCore128>(mode, a, p.how, st) : launch_dw_tiles<DwCore>(mode, a, p.how, st);
}

// The one-pass step of small batches (small_step.hpp).  Fn::operator()<S>() is called with the kernel for d dims and B
// rows; false if there is none: these six widths are the ones that are built (each is two kernels; 64, 192, 320, 640 and
// others would divide among waves in 32s too, and run as three passes), and 64 rows of 1024 dims with the waves' regions
// exceed the LDS.  Wherever there is one it is the faster than three passes: 1.24 to 4.1 times over 8 to 64 rows and 4,097 to
// 400,001 labels, least at 64 x 400,001 x 768 (768 -> 618 us); than G in one launch and the joint backward pass after it, but
// for 33 to 64 rows of 768 dims while W and M stay in the caches (see small_step).  384 dims and 64 rows take 12 waves of one block of dims:
// with 4 waves of three, 41 spills, 456 us at 64 x 400,001 instead of 307.
// large: W and M are more than the caches hold beside the rest (small_step_large); whole lines pay there for these (8, 32 and
// 64 rows x 90,001 to 2,000,003 labels: 1.02 to 1.10 times as fast with 768 dims, 0.98 to 1.08 with 1024, 1.02 to 1.15 with 512
// and 64 rows), not for 256 and 384 dims (0.84 to 1.12, most below 1) nor for 32 rows of 512 (0.87 to 1.11).
inline bool small_step_large(int64_t L, int64_t d) { return L * d * 4 > (int64_t)224 << 20; }
template <class Fn>
bool small_step_for(int64_t B, int64_t d, bool large, Fn&& fn) {
  if (B < 1 || B > SMALL_MAX_ROWS) return false;
  auto rows = [&](auto narrow, auto wide) {
    if (B <= 32) fn(narrow);
    else fn(wide);
    return true;
  };
  if (large && B > 32 && d == 512) { fn(SmallStep<8, 2, 4, true>{}); return true; }
  if (large && B <= 32 && d == 768) { fn(SmallStep<6, 4, 2, true>{}); return true; }
  if (large && B <= 32 && d == 1024) { fn(SmallStep<8, 4, 2, true>{}); return true; }
  switch (d) {
    case 128: return rows(SmallStep<4, 1, 2>{}, SmallStep<4, 1, 4>{});
    case 256: return rows(SmallStep<8, 1, 2>{}, SmallStep<8, 1, 4>{});
    case 384: return rows(SmallStep<4, 3, 2>{}, SmallStep<12, 1, 4>{});
    case 512: return rows(SmallStep<8, 2, 2>{}, SmallStep<8, 2, 4>{});
    case 768: return rows(SmallStep<8, 3, 2>{}, SmallStep<8, 3, 4>{});
    case 1024: if (B <= 32) { fn(SmallStep<8, 4, 2>{}); return true; } return false;
    default: return false;
  }
}
// The same for G alone: the weights are wanted again.
template <class Fn>
bool small_grad_for(int64_t B, int64_t d, Fn&& fn) {
  return small_step_for(B, d, false, [&](auto s) {
    if constexpr (!decltype(s)::LINES) fn(s);
  });
}
inline int small_step_tiles(int64_t L) { return ceil_div(round_up(L, 8), 32); }
// Workgroups, each with a partial dX of its own: as many as run at once.
template <class S>
int small_step_grid(int64_t L) {
  const int most = S::PER_CU * num_cus(), tiles = small_step_tiles(L);
  return tiles < most ? tiles : most;
}
// Bytes of the partial sums, 0 if there is no such kernel.
size_t small_step_ws_bytes(int64_t B, int64_t L, int64_t d) {
  size_t need = 0;
  if (L > 0) small_step_for(B, d, small_step_large(L, d), [&](auto s) { need = (size_t)small_step_grid<decltype(s)>(L) * B * d * 4; });
  return need;
}

// dX and dW (or the update) of a batch of up to 256 rows in one pass over the labels (back_step.hpp).  Fn::operator()<S>() is
// called with the kernel's sizes for B rows; false if there is none: more rows do not fit the LDS beside two images of their G.
// (Above 64
// rows it is the faster one at every size measured; see gradients_apart for the others.)
template <int MODE, class Fn>
bool back_step_for(int64_t B, Fn&& fn) {
  if (B < 1 || B > BACK_MAX_ROWS) return false;
  // what the addends and the update leave of the registers
  constexpr bool ADD = MODE == BACK_ADD, UPDATE = MODE == BACK_UPDATE;
  if (B <= 64) fn(BackStep<1, 2>{});
  else if (B <= 128) fn(BackStep<2, ADD ? 2 : 4>{});
  else if (B <= 192) fn(BackStep<3, ADD ? 2 : UPDATE ? 3 : 4>{});
  else fn(BackStep<4, ADD ? 0 : UPDATE ? 2 : 4>{});
  return true;
}
// Ranges of labels, one per workgroup: as many as there are CUs for their slices, in eighths for the XCDs; fewer where the
// labels or the workspace run out (8 at least).  On long label axes a range leaves a partial dX for each of its parts, so that
// no sum has more roundings than xfc_dx's (a tile's 64 labels are one addition here, four there).  Error of dX against float64
// by xfc_dx, by one chain of MFMAs per range, now: 199 rows x 131,072 x 768 2.8, 3.8, 1.7e-7, 256 x 320,001 x 384 3.4, 4.2,
// 1.9e-7, 5 x 60,007 x 3072 2.7, 5.6, 1.7e-7.
struct BackPlan { int ranges, parts; };
BackPlan back_plan(int64_t B, int64_t L, int64_t d, size_t ws_limit) {
  const int64_t slices = ceil_div(d, BACK_DIMS), per = num_cus() / (8 * slices), most = round_up(ceil_div(L, BACK_TILE), 8);
  int64_t ranges = 8 * (per > 1 ? per : 1);
  if (ranges > most) ranges = most;
  const size_t one = (size_t)B * (size_t)d * 4;
  while (ranges > 8 && (size_t)ranges * one > ws_limit) ranges -= 8;
  int tiles_m, tiles_n, sums, k_per_split;
  dx_plan((int)B, (int)d, (int)L, tiles_m, tiles_n, sums, k_per_split);
  int64_t parts = ceil_div(sums, 4 * ranges);
  while (parts > 1 && (size_t)(ranges * parts) * one > ws_limit) --parts;
  return {(int)ranges, (int)parts};
}
// The same for more rows (back_wide.hpp), the update only and widths of whole slices: there it is the faster at every size measured
// (whole steps of 257 to 512 rows x 1 to 2,812,281 labels x 128 to 3072 dims: 1.05 to 1.44 times, least at 400 x 131,073 x 1280,
// most at 320 x 400,001 x 128; the two passes read the weights and G twice).  With 193 to 256 rows the kernel above is (131,073
// x 768: 303 us by that one, 306 by this).
template <class Fn>
bool back_wide_for(int64_t B, int64_t d, Fn&& fn) {
  if (B <= BACK_MAX_ROWS || B > BACK_WIDE_ROWS || d % BACK_DIMS) return false;
  if (B <= 320) fn(BackWide<5>{});
  else if (B <= 384) fn(BackWide<6>{});
  else if (B <= 448) fn(BackWide<7>{});
  else fn(BackWide<8>{});
  return true;
}
// A workgroup per CU, and at least as many chains as xfc_dx has, for no longer ones.  (With fewer the error of dX grows, as the root
// of their lengths: 512 rows x 2,812,281 x 768, 128 of xfc_dx's, 126 here 1.01 times its 9.9e-7, 168 0.86; 300 x 2,080,392 x 1280, 125
// 1.015 and 150 0.92.  The longer reduction takes 0.4 % of that step, 7.22 -> 7.24 ms.)
BackPlan back_wide_plan(int64_t B, int64_t L, int64_t d) {
  const int64_t slices = d / BACK_DIMS, per = num_cus() / slices, tiles = ceil_div(L, BACK_TILE);
  const int64_t ranges = per < 1 ? 1 : per < tiles ? per : tiles;
  int tiles_m, tiles_n, sums, k_per_split;
  dx_plan((int)B, (int)d, (int)L, tiles_m, tiles_n, sums, k_per_split);
  return {(int)ranges, back_wide_parts((int)tiles, (int)ranges, sums)};
}
size_t back_ws_bytes(int64_t B, int64_t L, int64_t d) {
  if (B < 1 || B > BACK_WIDE_ROWS || L < 1 || d < 1 || (B > BACK_MAX_ROWS && d % BACK_DIMS)) return 0;
  const BackPlan p = B > BACK_MAX_ROWS ? back_wide_plan(B, L, d) : back_plan(B, L, d, ~(size_t)0);
  return (size_t)p.ranges * (size_t)p.parts * (size_t)B * (size_t)d * 4;
}
template <int MODE>
int launch_back(BackArgs a, float* dX, int64_t lddx, float scale, void* ws, size_t ws_bytes, hipStream_t st, bool* taken) {
  *taken = false;
  const BackPlan p = back_plan(a.B, a.L, a.d, ws_bytes);
  a.ranges = p.ranges;
  a.parts = p.parts;
  if (!ws || !aligned16(ws) || (size_t)a.ranges * a.B * a.d * 4 > ws_bytes) return XFC_OK;
  a.slices = ceil_div(a.d, BACK_DIMS);
  a.tiles = ceil_div(a.L, BACK_TILE);
  a.part = reinterpret_cast<float*>(ws);
  const bool lines = MODE == BACK_UPDATE ? whole_lines(a.W, a.ldw, a.d, 2) && whole_lines(a.Mo, a.ldm, a.d, 2) : whole_lines(a.out, a.ldo, a.d, 4);
  const StoreHow how = back_how(MODE == BACK_UPDATE, MODE == BACK_ADD, a.B, a.L, a.d, lines);
  int rc = XFC_OK;
  *taken = back_step_for<MODE>(a.B, [&](auto s) {
    using S = decltype(s);
    const dim3 g((unsigned)(a.slices * a.ranges)), b(S::NT);
    constexpr int SMALL = MODE == BACK_UPDATE ? THROUGH : CACHED;
    rc = how == PAST      ? launch_k<back_step_kernel<S, MODE, PAST>>(g, b, S::LDS_BYTES, st, a)
         : how == THROUGH ? launch_k<back_step_kernel<S, MODE, SMALL>>(g, b, S::LDS_BYTES, st, a)
                          : launch_k<back_step_kernel<S, MODE, CACHED>>(g, b, S::LDS_BYTES, st, a);
    if (rc) return;
    launch_dx_reduce(a.part, dX, lddx, a.B, a.d, a.ranges * a.parts, scale, 0.0f, st);
    rc = check_launch();
  });
  return rc;
}

int launch_back_wide(BackArgs a, float* dX, int64_t lddx, float scale, void* ws, size_t ws_bytes, hipStream_t st, bool* taken) {
  *taken = false;
  if (a.ldm != a.ldw || a.ldw >= (int64_t)1 << 27 || !ws || !aligned16(ws) || back_ws_bytes(a.B, a.L, a.d) > ws_bytes) return XFC_OK;
  int rc = XFC_OK;
  *taken = back_wide_for(a.B, a.d, [&](auto s) {
    using S = decltype(s);
    const BackPlan p = back_wide_plan(a.B, a.L, a.d);
    a.ranges = p.ranges;
    a.parts = p.parts;
    a.slices = a.d / BACK_DIMS;
    a.tiles = ceil_div(a.L, BACK_TILE);
    a.part = reinterpret_cast<float*>(ws);
    const dim3 g((unsigned)round_up(a.slices * a.ranges, 8)), b(S::NT);
    // Non-temporal loads where weights, momentum and G are more than the Infinity Cache holds (whole steps, without and with: 300
    // rows x 60,001 labels x 768 dims 147 and 152 us, 512 rows 184 and 182, 512 x 131,072 x 256 167 and 158).  There the forward pass has left the
    // caches the last labels' G and weights: those first (512 x 327,680 x 768 838 -> 825 us, 262,144 x 256 303 -> 286, 1,310,720 x
    // 768 3233 -> 3217), but not where these hold everything (300 x 60,001 x 768: 147 -> 160).
    // Non-temporal stores, which leave the cache to the weights that the next forward pass reads, in the other order, gain up to 2 % in steps
    // back to back and lose as much elsewhere.  Steps by themselves, each followed by 0.6 ms of matrix products over 96 MB, and each
    // waited for, with such stores and as it is: 512 x 131,073 x 768 364 and 370, 1002 and 991, 395 and 378 us; 512 x 180,001 x 768 489
    // and 483, 1116 and 1107, 509 and 495; 300 x 300,001 x 384 411 and 403, 1019 and 1011, 430 and 423.
    a.back = (int64_t)a.L * a.d * 4 + (int64_t)a.L * a.B * 2 > (int64_t)224 << 20;
    rc = a.back ? launch_k<back_wide_kernel<S, true>>(g, b, S::LDS_BYTES, st, a) : launch_k<back_wide_kernel<S, false>>(g, b, S::LDS_BYTES, st, a);
    if (rc) return;
    launch_dx_reduce(a.part, dX, lddx, a.B, a.d, a.ranges * a.parts, scale, 0.0f, st);
    rc = check_launch();
  });
  return rc;
}

int launch_generic(const void* in1, int64_t as0, int64_t as1, const void* in2, int64_t bs0, int64_t bs1, void* out,
                   int64_t os0, int64_t os1, int M, int N, int K, float alpha, float beta, int sigmoid, int out_half,
                   hipStream_t st) {
  if (M <= 0 || N <= 0) return XFC_OK;
  const int64_t tiles = (int64_t)ceil_div(M, GEN_T) * ceil_div(N, GEN_T);
  if (tiles > 0x7fffffff) return XFC_ERR_INVALID;
  hipLaunchKernelGGL(generic_gemm_kernel, dim3((unsigned)tiles), dim3(256), 0, st,
                     reinterpret_cast<const half_t*>(in1), as0, as1, reinterpret_cast<const half_t*>(in2), bs0, bs1,
                     out, os0, os1, M, N, K, alpha, beta, sigmoid, out_half);
  return check_launch();
}

template <int RB>
int launch_score_small(ScoreArgs a, hipStream_t st) {
  constexpr int NW = SCORE_SMALL_WAVES;
  const int64_t most = (int64_t)2 * num_cus(), units = ceil_div(a.N, SCORE_SMALL_BLOCK), waves = most * NW;
  // Units in a row for a wave: a row's maxima are then stored 8 or 16 bytes at a time (32 rows x 700,001 labels x 768: 217 -> 208
  // us), as long as that leaves the longest wave's work what it is, or with 32 rows to store for a tenth more.
  a.run = 1;
  for (int run : {2, 4})
    if (10 * run * ceil_div(units, run * waves) <= (RB == 1 ? 10 : 11) * ceil_div(units, waves)) a.run = run;
  const int64_t want = ceil_div(units, a.run * NW);
  // (the limit is raised once, for any width)
  const hipError_t e = raise_lds_limit<score_small_kernel<RB>>(FULL_LDS);
  if (e != hipSuccess) {
    fprintf(stderr, "xfc: cannot raise the dynamic LDS limit to %d bytes: %s\n", FULL_LDS, hipGetErrorString(e));
    return XFC_ERR_HIP;
  }
  return launch_k<score_small_kernel<RB>>(dim3((unsigned)(want < most ? want : most)), dim3(64 * NW), (int)score_small_lds<RB>(a.K), st, a);
}

struct SelArgs {
  const half_t* logits; int64_t ldl; int L; int64_t numy; int K; int stride;
  const half_t* bmax; int64_t ldb; int n_blocks; float* out_v; int64_t* out_i;
};
template <int CAP>
int launch_select(int rows, const SelArgs& a, hipStream_t st) {
  constexpr int LDS = (int)sizeof(SelLds<CAP>);
  static_assert(LDS <= 160 * 1024, "LDS budget");
  const hipError_t e = raise_lds_limit<topk_select_kernel<CAP>>(LDS);
  if (e != hipSuccess) {
    fprintf(stderr, "xfc: cannot raise the dynamic LDS limit to %d bytes: %s\n", LDS, hipGetErrorString(e));
    return XFC_ERR_HIP;
  }
  hipLaunchKernelGGL(topk_select_kernel<CAP>, dim3((unsigned)rows), dim3(SEL_THREADS), LDS, st, a.logits, a.ldl, a.L, a.numy,
                     a.K, a.stride, a.bmax, a.ldb, a.n_blocks, a.out_v, a.out_i);
  return check_launch();
}

bool dims_ok(int64_t v) { return v >= 0 && v <= 0x7fffffff; }

}  // namespace

extern "C" {

const char* xfc_strerror(int code) {
  switch (code) {
    case XFC_OK: return "ok";
    case XFC_ERR_INVALID: return "invalid argument (null pointer, negative or oversized dimension)";
    case XFC_ERR_LAYOUT: return "unsupported operand layout: expected row x column (sigmoid), column x row, or row x row";
    case XFC_ERR_ALIGN: return "operand pointer or leading dimension not aligned to 16 bytes";
    case XFC_ERR_WORKSPACE: return "workspace missing or too small";
    case XFC_ERR_HIP: return "HIP runtime error";
    case XFC_ERR_SHAPE: return "operand shapes do not agree";
    case XFC_ERR_LIMIT: return "problem larger than the fixed capacity of this entry point";
    default: return "unknown error";
  }
}

int xfc_abi_version(void) { return XFC_ABI_VERSION; }

int xfc_init(void) {
  hipError_t e = hipSuccess;
  auto keep = [&](hipError_t r) { if (e == hipSuccess) e = r; };
  auto wide_limits = [&](auto core_tag) {
    using C = typename decltype(core_tag)::type;
    keep(raise_lds_limit<fwd_wide_kernel<C, FWD_SIGMOID_PLAIN, false, true>>(C::LDS_BYTES));
    keep(raise_lds_limit<fwd_wide_kernel<C, FWD_SIGMOID, true>>(C::LDS_BYTES));
    keep(raise_lds_limit<fwd_wide_kernel<C, FWD_SIGMOID, false>>(C::LDS_BYTES));
    keep(raise_lds_limit<fwd_wide_kernel<C, FWD_SIGMOID_PLAIN, false>>(C::LDS_BYTES));
    keep(raise_lds_limit<fwd_wide_kernel<C, FWD_LINEAR, false>>(C::LDS_BYTES));
    keep(raise_lds_limit<fwd_wide_kernel<C, FWD_LINEAR, false, false, true>>(C::LDS_BYTES));
  };
  wide_limits(std::type_identity<FwdWide>{});
  wide_limits(std::type_identity<FwdWide128>{});
  keep(raise_lds_limit<score_wide_kernel<ScoreWide>>(ScoreWide::LDS_BYTES));
  keep(raise_lds_limit<score_wide_kernel<ScoreWide128>>(ScoreWide128::LDS_BYTES));
  keep(raise_lds_limit<topk_list_kernel<ListCore>>(TopkLds<ListCore>::BYTES));
  keep(raise_lds_limit<topk_list_kernel<ListCore128>>(TopkLds<ListCore128>::BYTES));
  keep(raise_lds_limit<topk_list_kernel<ListCore64>>(TopkLds<ListCore64>::BYTES));
  keep(raise_lds_limit<dx_wide_kernel<CACHED>>(DxWide::LDS_BYTES));
  keep(raise_lds_limit<dx_wide_kernel<THROUGH>>(DxWide::LDS_BYTES));
  auto small_limits = [&](auto core_tag, auto dx_tag) {
    using C = typename decltype(core_tag)::type;
    using D = typename decltype(dx_tag)::type;
    constexpr int LDS = FwdLds<C>::BYTES;
    keep(raise_lds_limit<fwd_kernel<C, FWD_SIGMOID_PLAIN, false, true>>(LDS));
    keep(raise_lds_limit<fwd_kernel<C, FWD_SIGMOID, true>>(LDS));
    keep(raise_lds_limit<fwd_kernel<C, FWD_SIGMOID, false>>(LDS));
    keep(raise_lds_limit<fwd_kernel<C, FWD_SIGMOID_PLAIN, false>>(LDS));
    keep(raise_lds_limit<fwd_kernel<C, FWD_LINEAR, false>>(LDS));
    keep(raise_lds_limit<fwd_kernel<C, FWD_LINEAR, false, false, true>>(LDS));
    keep(raise_lds_limit<dx_kernel<D, CACHED>>(D::LDS_BYTES));
    keep(raise_lds_limit<dx_kernel<D, THROUGH>>(D::LDS_BYTES));
  };
  small_limits(std::type_identity<FwdCore>{}, std::type_identity<DxCore>{});
  small_limits(std::type_identity<FwdCore64>{}, std::type_identity<DxCore64>{});
  for (int64_t rows : {32, 64})
    for (int64_t d : {128, 256, 384, 512, 768, 1024})
      for (bool large : {false, true}) {
        small_step_for(rows, d, large, [&](auto s) { keep(raise_lds_limit<small_step_kernel<decltype(s)>>(decltype(s)::LDS_BYTES)); });
        small_grad_for(rows, d, [&](auto s) { keep(raise_lds_limit<small_step_kernel<decltype(s), false>>(decltype(s)::LDS_BYTES)); });
      }
  keep(raise_lds_limit<score_small_kernel<1>>(FULL_LDS));
  keep(raise_lds_limit<score_small_kernel<2>>(FULL_LDS));
  auto back_limits = [&](auto mode) {
    constexpr int MODE = decltype(mode)::value;
    for (int64_t rows : {64, 128, 192, 256})
      back_step_for<MODE>(rows, [&](auto s) {
        using S = decltype(s);
        keep(raise_lds_limit<back_step_kernel<S, MODE, CACHED>>(S::LDS_BYTES));
        keep(raise_lds_limit<back_step_kernel<S, MODE, PAST>>(S::LDS_BYTES));
        if constexpr (MODE == BACK_UPDATE) keep(raise_lds_limit<back_step_kernel<S, MODE, THROUGH>>(S::LDS_BYTES));
      });
  };
  for (int64_t rows : {320, 384, 448, 512})
    back_wide_for(rows, BACK_DIMS, [&](auto s) {
      using S = decltype(s);
      keep(raise_lds_limit<back_wide_kernel<S, false>>(S::LDS_BYTES));
      keep(raise_lds_limit<back_wide_kernel<S, true>>(S::LDS_BYTES));
    });
  back_limits(std::integral_constant<int, BACK_UPDATE>{});
  back_limits(std::integral_constant<int, BACK_OUT>{});
  back_limits(std::integral_constant<int, BACK_ADD>{});
  keep(raise_lds_limit<topk_select_kernel<SEL_CAP_SMALL>>((int)sizeof(SelLds<SEL_CAP_SMALL>)));
  keep(raise_lds_limit<topk_select_kernel<SEL_CAP_LARGE>>((int)sizeof(SelLds<SEL_CAP_LARGE>)));
  auto dw_limits = [&](auto core_tag, auto mode) {
    using C = typename decltype(core_tag)::type;
    constexpr int MODE = decltype(mode)::value, LDS = DwLds<C>::BYTES;
    keep(raise_lds_limit<dw_kernel<C, MODE, THROUGH>>(LDS));
    keep(raise_lds_limit<dw_kernel<C, MODE, PAST>>(LDS));
    keep(raise_lds_limit<dw_kernel<C, MODE, CACHED>>(LDS));
  };
  auto dw_all_limits = [&](auto core_tag) {
    dw_limits(core_tag, std::integral_constant<int, DW_UPDATE>{});
    dw_limits(core_tag, std::integral_constant<int, DW_OUT>{});
    dw_limits(core_tag, std::integral_constant<int, DW_UPDATE_MASTER>{});
  };
  dw_all_limits(std::type_identity<DwCore>{});
  dw_all_limits(std::type_identity<DwCore128>{});
  (void)num_cus();
  if (static_scratch_ptr() == nullptr) return XFC_ERR_HIP;
  if (e != hipSuccess) {
    fprintf(stderr, "xfc: xfc_init failed: %s\n", hipGetErrorString(e));
    return XFC_ERR_HIP;
  }
  return XFC_OK;
}

size_t xfc_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (!dims_ok(M) || !dims_ok(N) || !dims_ok(K)) return 0;
  int tm, tn, s, kps;
  dx_plan((int)M, (int)N, (int)K, tm, tn, s, kps);
  return (size_t)s * M * N * 4;
}

int xfc_gemm(const void* in1, int64_t in1_rows, int64_t in1_cols, int64_t in1_s0, int64_t in1_s1, const void* in2,
             int64_t in2_rows, int64_t in2_cols, int64_t in2_s0, int64_t in2_s1, void* out, int64_t out_rows,
             int64_t out_cols, int64_t out_s0, int64_t out_s1, float alpha, float beta, int apply_sigmoid,
             void* workspace, size_t workspace_bytes, void* stream) {
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t M = out_rows, N = out_cols, K = in2_rows;
  if (!dims_ok(M) || !dims_ok(N) || !dims_ok(K)) return XFC_ERR_INVALID;
  if (in1_rows != M || in1_cols != K || in2_cols != N) return XFC_ERR_SHAPE;
  if (M == 0 || N == 0) return XFC_OK;
  if (!in1 || !in2 || !out) return XFC_ERR_INVALID;
  const bool a_row = in1_s1 == 1, a_col = in1_s0 == 1, b_row = in2_s1 == 1, b_col = in2_s0 == 1;
  if (apply_sigmoid) {
    // out(fp16) = sigmoid(alpha * in1 . in2 + beta * out), in1 row-major, in2 column-major
    if (!(a_row && b_col)) return XFC_ERR_LAYOUT;
    const bool fast = out_s1 == 1 && out_s0 % 8 == 0 && aligned16(out) && in1_s0 % 8 == 0 && in2_s1 % 8 == 0 &&
                      K % 8 == 0 && aligned16(in1) && aligned16(in2) && K > 0;
    if (fast)
      return launch_fwd(fwd_plan(M, N, K, false, num_cus()), FWD_SIGMOID, (const half_t*)in1, in1_s0, (const half_t*)in2, in2_s1, (half_t*)out,
                        out_s0, (int)M, (int)N, (int)K, (int)N, alpha, beta, st);
    return launch_generic(in1, in1_s0, in1_s1, in2, in2_s0, in2_s1, out, out_s0, out_s1, (int)M, (int)N, (int)K, alpha,
                          beta, 1, 1, st);
  }
  if (a_col && b_row) {
    // out(fp32) = alpha * in1 . in2 + beta * out, in1 column-major (G^T view), in2 row-major (X)
    const bool fast = out_s1 == 1 && out_s0 % 4 == 0 && aligned16(out) && in1_s1 % 8 == 0 && in2_s0 % 8 == 0 &&
                      N % 8 == 0 && M % 8 == 0 && aligned16(in1) && aligned16(in2) && K > 0;
    if (fast) {
      DwArgs a = {};
      a.G = (const half_t*)in1; a.ldg = in1_s1; a.X = (const half_t*)in2; a.ldx = in2_s0;
      a.M = (int)M; a.N = (int)N; a.K = (int)K; a.g_cols = (int)round_up(M, 8);
      a.out = (float*)out; a.ldo = out_s0; a.alpha = alpha; a.beta = beta;
      return launch_dw(DW_OUT, a, st);
    }
    return launch_generic(in1, in1_s0, in1_s1, in2, in2_s0, in2_s1, out, out_s0, out_s1, (int)M, (int)N, (int)K, alpha,
                          beta, 0, 0, st);
  }
  if (a_row && b_row) {
    // out(fp32) = alpha * in1 . in2 + beta * out, both row-major: contraction over in1's columns
    const bool fast = out_s1 == 1 && in1_s0 % 8 == 0 && in2_s0 % 8 == 0 && N % 8 == 0 && K % 8 == 0 &&
                      aligned16(in1) && aligned16(in2) && K > 0;
    if (fast) {
      return launch_dx((const half_t*)in1, in1_s0, (const half_t*)in2, in2_s0, (float*)out, out_s0, (int)M, (int)N,
                       (int)K, alpha, beta, workspace, workspace_bytes, st);
    }
    return launch_generic(in1, in1_s0, in1_s1, in2, in2_s0, in2_s1, out, out_s0, out_s1, (int)M, (int)N, (int)K, alpha,
                          beta, 0, 0, st);
  }
  return XFC_ERR_LAYOUT;
}

int xfc_logits(const void* X, int64_t ldx, const void* W, int64_t ldw, void* out, int64_t ldo, int64_t B, int64_t L,
               int64_t d, void* stream) {
  if (!dims_ok(B) || !dims_ok(L) || !dims_ok(d)) return XFC_ERR_INVALID;
  if (B == 0 || L == 0) return XFC_OK;
  if (!X || !W || !out || d <= 0) return XFC_ERR_INVALID;
  if (ldx % 8 || ldw % 8 || ldo % 8 || d % 8 || !aligned16(X) || !aligned16(W) || !aligned16(out))
    return XFC_ERR_ALIGN;
  if (ldo < L) return XFC_ERR_SHAPE;
  return launch_fwd(fwd_plan(B, L, d, false, num_cus()), FWD_LINEAR, (const half_t*)X, ldx, (const half_t*)W, ldw, (half_t*)out, ldo, (int)B,
                    (int)L, (int)d, (int)L, 1.0f, 0.0f, reinterpret_cast<hipStream_t>(stream));
}

size_t xfc_fwd_grad_workspace_bytes(int64_t L, int64_t nnz) {
  if (!dims_ok(L) || nnz < 0) return 0;
  return fwd_ws_bytes(nnz);
}

// What small_step_kernel reads for G.
static SmallArgs small_args(const void* X, int64_t ldx, const void* W, int64_t ldw, const int32_t* rowptr, const int32_t* colidx,
                            const int64_t* pos_x, const int64_t* pos_y, int64_t nnz, void* G, int64_t ldg, int64_t B, int64_t L) {
  SmallArgs a = {};
  a.X = (const half_t*)X; a.ldx = ldx; a.W = (half_t*)const_cast<void*>(W); a.ldw = ldw;
  a.G = (half_t*)G; a.ldg = ldg;
  a.rowptr = rowptr; a.colidx = colidx; a.pos_x = pos_x; a.pos_y = pos_y;
  a.nnz = (int)nnz; a.B = (int)B; a.L = (int)L; a.n_store = (int)round_up(L, 8); a.tiles = small_step_tiles(L);
  return a;
}

// G of a small batch and its positives in one launch, if there is such a kernel for the call (whose arguments have been
// checked): no loss, no more pairs than the workgroups' threads hold.  XFC_OK with *taken false otherwise.  It stands as long as
// it is the faster one: 32 rows x 131,072 x 768 41 -> 33 us and x 4,097 launch-bound, 16 -> 13, but x 320,001 97 -> 101; with 64 rows
// its two barriers a tile weigh more, x 20,011 16 -> 13 but x 60,007 21 -> 25, and at 128 dims x 100,003 16.6 -> 15.1 but x 131,072
// 16.4 -> 17.9.
static int small_grad(const void* X, int64_t ldx, const void* W, int64_t ldw, const int32_t* rowptr, const int32_t* colidx,
                      const int64_t* pos_x, const int64_t* pos_y, int64_t nnz, void* G, int64_t ldg, int64_t B, int64_t L, int64_t d,
                      const float* loss, hipStream_t st, bool* taken) {
  *taken = false;
  if (loss || B > SMALL_MAX_ROWS || nnz > SMALL_MAX_PAIRS) return XFC_OK;
  if (B <= 32 ? L * d > (int64_t)160 << 20 : L * d > (int64_t)16 << 20 || L > 100 << 10) return XFC_OK;
  const SmallArgs a = small_args(X, ldx, W, ldw, rowptr, colidx, pos_x, pos_y, nnz, G, ldg, B, L);
  int rc = XFC_OK;
  *taken = small_grad_for(B, d, [&](auto s) {
    using S = decltype(s);
    rc = launch_k<small_step_kernel<S, false>>(dim3((unsigned)small_step_grid<S>(L)), dim3(S::NT), S::LDS_BYTES, st, a);
  });
  return rc;
}

static int fwd_grad_impl(const void* X, int64_t ldx, const void* W, int64_t ldw, const int32_t* rowptr,
                         const int32_t* colidx, const int64_t* pos_x, const int64_t* pos_y, int64_t nnz, void* G,
                         int64_t ldg, int64_t B, int64_t L, int64_t d, float* loss, void* ws, size_t ws_bytes,
                         hipStream_t st) {
  if (!dims_ok(B) || !dims_ok(L) || !dims_ok(d) || nnz < 0 || nnz > 0x7fffffff) return XFC_ERR_INVALID;
  if (B == 0 || L == 0) return XFC_OK;
  if (!X || !W || !G || d <= 0) return XFC_ERR_INVALID;
  if (nnz > 0 && !((rowptr && colidx) || (pos_x && pos_y))) return XFC_ERR_INVALID;
  if (ldx % 8 || ldw % 8 || ldg % 8 || d % 8 || !aligned16(X) || !aligned16(W) || !aligned16(G))
    return XFC_ERR_ALIGN;
  if (ldg < L) return XFC_ERR_SHAPE;
  if (!ws || ws_bytes < fwd_ws_bytes(nnz)) return XFC_ERR_WORKSPACE;
  bool taken;
  if (int rc0 = small_grad(X, ldx, W, ldw, rowptr, colidx, pos_x, pos_y, nnz, G, ldg, B, L, d, loss, st, &taken); taken) return rc0;
  const LossPart loss_part = loss ? loss_part_of(ws) : NO_LOSS;
  float* loss_pos = loss ? reinterpret_cast<float*>(reinterpret_cast<unsigned char*>(ws) + LOSS_PART_BYTES) : nullptr;
  // label columns L .. round_up(L, 8) are written as zero so that G can be read in 16-byte
  // pieces along the label axis by the dX and dW kernels (ldg is a multiple of 8, so they exist)
  const int64_t n_store = round_up(L, 8);
  const FwdPlan plan = fwd_plan(B, n_store, d, loss != nullptr, num_cus());
  int rc = launch_fwd(plan, FWD_SIGMOID, (const half_t*)X, ldx, (const half_t*)W, ldw, (half_t*)G, ldg, (int)B, (int)L, (int)d,
                      (int)n_store, 1.0f, 0.0f, st, loss_part);
  if (rc) return rc;
  if (nnz > 0) {
    const int64_t blocks = ceil_div(nnz, 4) < 16384 ? ceil_div(nnz, 4) : 16384;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, st, (const half_t*)X, ldx, (const half_t*)W, ldw,
                         rowptr, colidx, pos_x, pos_y, nnz, (int)B, L, (int)d, (half_t*)G, ldg, loss_pos);
    };
    if (!loss) launch(positives_kernel<POS_G>);
    else if (plan.tile == FWD_WIDE || plan.tile == FWD_WIDE128) launch(positives_kernel<POS_LOSS_WIDE>);
    else launch(positives_kernel<POS_LOSS>);
    if ((rc = check_launch())) return rc;
  }
  if (loss) {
    const int64_t first = fwd_grid(plan, B, num_cus(), loss_part.places), rest = fwd_rest_grid(plan, B, n_store, num_cus(), loss_part.places);
    hipLaunchKernelGGL(loss_reduce_kernel, dim3(1), dim3(1024), 0, st, (const double*)loss_part.at, (int)(first > rest ? first : rest),
                       (const float*)loss_pos, nnz, loss);
    return check_launch();
  }
  return XFC_OK;
}

int xfc_fwd_grad_csr(const void* X, int64_t ldx, const void* W, int64_t ldw, const int32_t* rowptr,
                     const int32_t* colidx, void* G, int64_t ldg, int64_t B, int64_t L, int64_t d, int64_t nnz,
                     float* loss, void* workspace, size_t workspace_bytes, void* stream) {
  if (B > 0 && !rowptr) return XFC_ERR_INVALID;
  return fwd_grad_impl(X, ldx, W, ldw, rowptr, colidx, nullptr, nullptr, nnz, G, ldg, B, L, d, loss, workspace,
                       workspace_bytes, reinterpret_cast<hipStream_t>(stream));
}

int xfc_fwd_grad_csr_static(const void* X, int64_t ldx, const void* W, int64_t ldw, const int32_t* rowptr,
                            const int32_t* colidx, void* G, int64_t ldg, int64_t B, int64_t L, int64_t d, int64_t nnz,
                            float* loss, void* stream) {
  if (B > 0 && !rowptr) return XFC_ERR_INVALID;
  if (!dims_ok(L) || nnz < 0) return XFC_ERR_INVALID;
  if (fwd_ws_bytes(nnz) > (size_t)XFC_STATIC_SCRATCH_BYTES) {
    fprintf(stderr, "xfc_fwd_grad_csr_static: L = %lld labels with %lld positives need %zu bytes of scratch, the static "
                    "buffer holds %d; use xfc_fwd_grad_csr with a caller workspace\n",
            (long long)L, (long long)nnz, fwd_ws_bytes(nnz), XFC_STATIC_SCRATCH_BYTES);
    return XFC_ERR_LIMIT;
  }
  void* scratch = static_scratch_ptr();
  if (scratch == nullptr) return XFC_ERR_HIP;
  // what the loss reduction reads is written by this call first, so nothing of the previous call's contents
  // survives into this one
  return fwd_grad_impl(X, ldx, W, ldw, rowptr, colidx, nullptr, nullptr, nnz, G, ldg, B, L, d, loss, scratch,
                       (size_t)XFC_STATIC_SCRATCH_BYTES, reinterpret_cast<hipStream_t>(stream));
}

int xfc_fwd_grad_coo(const void* X, int64_t ldx, const void* W, int64_t ldw, const int64_t* pos_x, const int64_t* pos_y,
                     int64_t nnz, void* G, int64_t ldg, int64_t B, int64_t L, int64_t d, float* loss, void* workspace,
                     size_t workspace_bytes, void* stream) {
  if (nnz > 0 && !(pos_x && pos_y)) return XFC_ERR_INVALID;
  return fwd_grad_impl(X, ldx, W, ldw, nullptr, nullptr, pos_x, pos_y, nnz, G, ldg, B, L, d, loss, workspace, workspace_bytes,
                       reinterpret_cast<hipStream_t>(stream));
}

size_t xfc_dx_workspace_bytes(int64_t B, int64_t L, int64_t d) { return xfc_gemm_workspace_bytes(B, d, L); }

int xfc_dx(const void* G, int64_t ldg, const void* W, int64_t ldw, float* dX, int64_t lddx, int64_t B, int64_t L,
           int64_t d, float scale, void* workspace, size_t workspace_bytes, void* stream) {
  if (!dims_ok(B) || !dims_ok(L) || !dims_ok(d)) return XFC_ERR_INVALID;
  if (B == 0 || d == 0) return XFC_OK;
  if (!G || !W || !dX) return XFC_ERR_INVALID;
  if (ldg % 8 || ldw % 8 || d % 8 || !aligned16(G) || !aligned16(W)) return XFC_ERR_ALIGN;
  if (ldg < round_up(L, 8)) return XFC_ERR_SHAPE;
  return launch_dx((const half_t*)G, ldg, (const half_t*)W, ldw, dX, lddx, (int)B, (int)d, (int)L, scale, 0.0f,
                   workspace, workspace_bytes, reinterpret_cast<hipStream_t>(stream));
}

int xfc_dw_update(const void* G, int64_t ldg, const void* X, int64_t ldx, void* W, int64_t ldw, void* Mo, int64_t ldm,
                  int64_t B, int64_t L, int64_t d, float lr, float momentum, float weight_decay, float* dW_out,
                  int64_t ld_dw, void* stream) {
  if (!dims_ok(B) || !dims_ok(L) || !dims_ok(d)) return XFC_ERR_INVALID;
  if (L == 0 || d == 0 || B == 0) return XFC_OK;  // an empty batch is not a step: W and M stay as they are
  if (!G || !X || !W || !Mo) return XFC_ERR_INVALID;
  if (ldg % 8 || ldx % 8 || ldw % 8 || ldm % 8 || d % 8 || !aligned16(G) || !aligned16(X) || !aligned16(W) ||
      !aligned16(Mo))
    return XFC_ERR_ALIGN;
  if (dW_out && (ld_dw % 4 || !aligned16(dW_out))) return XFC_ERR_ALIGN;
  if (ldg < round_up(L, 8)) return XFC_ERR_SHAPE;
  DwArgs a = {};
  a.G = (const half_t*)G; a.ldg = ldg; a.X = (const half_t*)X; a.ldx = ldx;
  a.M = (int)L; a.N = (int)d; a.K = (int)B; a.g_cols = (int)round_up(L, 8);
  a.Wt = (half_t*)W; a.ldw = ldw; a.Mo = (half_t*)Mo; a.ldm = ldm;
  a.lr = lr; a.mu = momentum; a.wd = weight_decay; a.dw_dump = dW_out; a.ld_dump = ld_dw;
  return launch_dw(DW_UPDATE, a, reinterpret_cast<hipStream_t>(stream));
}

int xfc_dw_update_master(const void* G, int64_t ldg, const void* X, int64_t ldx, float* W32, int64_t ldw32, float* M32,
                         int64_t ldm32, void* W16, int64_t ldw16, int64_t B, int64_t L, int64_t d, float lr,
                         float momentum, float weight_decay, float* dW_out, int64_t ld_dw, void* stream) {
  if (!dims_ok(B) || !dims_ok(L) || !dims_ok(d)) return XFC_ERR_INVALID;
  if (L == 0 || d == 0 || B == 0) return XFC_OK;  // an empty batch is not a step
  if (!G || !X || !W32 || !M32 || !W16) return XFC_ERR_INVALID;
  if (ldg % 8 || ldx % 8 || ldw16 % 8 || ldw32 % 4 || ldm32 % 4 || d % 8 || !aligned16(G) || !aligned16(X) ||
      !aligned16(W32) || !aligned16(M32) || !aligned16(W16))
    return XFC_ERR_ALIGN;
  if (dW_out && (ld_dw % 4 || !aligned16(dW_out))) return XFC_ERR_ALIGN;
  if (ldg < round_up(L, 8)) return XFC_ERR_SHAPE;
  DwArgs a = {};
  a.G = (const half_t*)G; a.ldg = ldg; a.X = (const half_t*)X; a.ldx = ldx;
  a.M = (int)L; a.N = (int)d; a.K = (int)B; a.g_cols = (int)round_up(L, 8);
  a.Wt = (half_t*)W16; a.ldw = ldw16; a.W32 = W32; a.ldw32 = ldw32; a.M32 = M32; a.ldm32 = ldm32;
  a.lr = lr; a.mu = momentum; a.wd = weight_decay; a.dw_dump = dW_out; a.ld_dump = ld_dw;
  return launch_dw(DW_UPDATE_MASTER, a, reinterpret_cast<hipStream_t>(stream));
}

int xfc_sgd_momentum_master(float* W32, float* M32, void* W16, const float* grad, int64_t count, float lr, float momentum,
                            float weight_decay, void* stream) {
  if (count < 0) return XFC_ERR_INVALID;
  if (count == 0) return XFC_OK;
  if (!W32 || !M32 || !W16 || !grad) return XFC_ERR_INVALID;
  if (count % 8 || !aligned16(W32) || !aligned16(M32) || !aligned16(W16) || !aligned16(grad)) return XFC_ERR_ALIGN;
  const int64_t n8 = count / 8;
  hipLaunchKernelGGL(sgd_momentum_master_kernel, dim3((unsigned)ceil_div(n8, 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), W32, M32, (half_t*)W16, grad, n8, lr, momentum, weight_decay);
  return check_launch();
}

int xfc_dw(const void* G, int64_t ldg, const void* X, int64_t ldx, float* grad, int64_t ld_grad, int64_t B, int64_t L,
           int64_t d, float beta, void* stream) {
  if (!dims_ok(B) || !dims_ok(L) || !dims_ok(d)) return XFC_ERR_INVALID;
  if (L == 0 || d == 0) return XFC_OK;
  if (B == 0 && beta == 1.0f) return XFC_OK;  // an empty micro-batch adds nothing
  if (B == 0) return XFC_ERR_INVALID;          // beta != 1 with no rows would only rescale grad: not a dW call
  if (!G || !X || !grad) return XFC_ERR_INVALID;
  if (ldg % 8 || ldx % 8 || d % 8 || ld_grad % 4 || !aligned16(G) || !aligned16(X) || !aligned16(grad))
    return XFC_ERR_ALIGN;
  if (ldg < round_up(L, 8)) return XFC_ERR_SHAPE;
  DwArgs a = {};
  a.G = (const half_t*)G; a.ldg = ldg; a.X = (const half_t*)X; a.ldx = ldx;
  a.M = (int)L; a.N = (int)d; a.K = (int)B; a.g_cols = (int)round_up(L, 8);
  a.out = grad; a.ldo = ld_grad; a.alpha = 1.0f; a.beta = beta;
  return launch_dw(DW_OUT, a, reinterpret_cast<hipStream_t>(stream));
}

int xfc_sgd_momentum(void* W, void* Mo, const float* grad, int64_t count, float lr, float momentum, float weight_decay,
                     void* stream) {
  if (count < 0) return XFC_ERR_INVALID;
  if (count == 0) return XFC_OK;
  if (!W || !Mo || !grad) return XFC_ERR_INVALID;
  if (count % 8 || !aligned16(W) || !aligned16(Mo) || !aligned16(grad)) return XFC_ERR_ALIGN;
  const int64_t n8 = count / 8;
  hipLaunchKernelGGL(sgd_momentum_kernel, dim3((unsigned)ceil_div(n8, 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), (half_t*)W, (half_t*)Mo, grad, n8, lr, momentum,
                     weight_decay);
  return check_launch();
}

// Both gradients of a batch; what the one pass does not take runs as two, which also report what is wrong with a call.
static bool back_ok(const void* G, int64_t ldg, const void* X, int64_t ldx, const void* W, int64_t ldw, const void* dX, int64_t B,
                    int64_t L, int64_t d, int64_t rows = BACK_MAX_ROWS) {
  return dims_ok(B) && dims_ok(L) && dims_ok(d) && B >= 1 && B <= rows && L >= 1 && d >= 8 && G && X && W && dX &&
         ldg % 8 == 0 && ldg < (int64_t)1 << 27 && ldx % 8 == 0 && ldw % 8 == 0 && d % 8 == 0 && aligned16(G) && aligned16(X) && aligned16(W) &&
         ldg >= round_up(L, 8);
}
static BackArgs back_args(const void* G, int64_t ldg, const void* X, int64_t ldx, const void* W, int64_t ldw, int64_t B, int64_t L,
                          int64_t d) {
  BackArgs a = {};
  a.G = (const half_t*)G; a.ldg = ldg; a.X = (const half_t*)X; a.ldx = ldx; a.W = (half_t*)const_cast<void*>(W); a.ldw = ldw;
  a.B = (int)B; a.L = (int)L; a.d = (int)d;
  return a;
}

int xfc_dx_dw_update(const void* G, int64_t ldg, const void* X, int64_t ldx, void* W, int64_t ldw, void* Mo, int64_t ldm, float* dX,
                     int64_t lddx, int64_t B, int64_t L, int64_t d, float lr, float momentum, float weight_decay, float scale,
                     void* workspace, size_t workspace_bytes, void* stream) {
  if (back_ok(G, ldg, X, ldx, W, ldw, dX, B, L, d, BACK_WIDE_ROWS) && Mo && ldm % 8 == 0 && aligned16(Mo)) {
    BackArgs a = back_args(G, ldg, X, ldx, W, ldw, B, L, d);
    a.Mo = (half_t*)Mo; a.ldm = ldm; a.lr = lr; a.mu = momentum; a.wd = weight_decay;
    bool taken;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int rc = B > BACK_MAX_ROWS ? launch_back_wide(a, dX, lddx, scale, workspace, workspace_bytes, st, &taken)
                                     : launch_back<BACK_UPDATE>(a, dX, lddx, scale, workspace, workspace_bytes, st, &taken);
    if (taken) return rc;
  }
  const int rc = xfc_dx(G, ldg, W, ldw, dX, lddx, B, L, d, scale, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return xfc_dw_update(G, ldg, X, ldx, W, ldw, Mo, ldm, B, L, d, lr, momentum, weight_decay, nullptr, 0, stream);
}

int xfc_dx_dw(const void* G, int64_t ldg, const void* X, int64_t ldx, const void* W, int64_t ldw, float* grad, int64_t ld_grad,
              float* dX, int64_t lddx, int64_t B, int64_t L, int64_t d, float beta, float scale, void* workspace,
              size_t workspace_bytes, void* stream) {
  const bool apart = dims_ok(B) && dims_ok(L) && dims_ok(d) && d > 0 && gradients_apart(B, L, d, beta != 0.f, num_cus());
  if (!apart && back_ok(G, ldg, X, ldx, W, ldw, dX, B, L, d) && grad && ld_grad % 4 == 0 && aligned16(grad)) {
    BackArgs a = back_args(G, ldg, X, ldx, W, ldw, B, L, d);
    a.out = grad; a.ldo = ld_grad; a.beta = beta;
    bool taken;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int rc = beta != 0.f ? launch_back<BACK_ADD>(a, dX, lddx, scale, workspace, workspace_bytes, st, &taken)
                               : launch_back<BACK_OUT>(a, dX, lddx, scale, workspace, workspace_bytes, st, &taken);
    if (taken) return rc;
  }
  const int rc = xfc_dx(G, ldg, W, ldw, dX, lddx, B, L, d, scale, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return xfc_dw(G, ldg, X, ldx, grad, ld_grad, B, L, d, beta, stream);
}

size_t xfc_step_workspace_bytes(int64_t B, int64_t L, int64_t d, int64_t nnz) {
  const size_t dx = xfc_dx_workspace_bytes(B, L, d), small = dims_ok(B) && dims_ok(L) && dims_ok(d) ? small_step_ws_bytes(B, L, d) : 0;
  const size_t back = dims_ok(B) && dims_ok(L) && dims_ok(d) ? back_ws_bytes(B, L, d) : 0, most = dx > small ? dx : small;
  return (size_t)round_up(xfc_fwd_grad_workspace_bytes(L, nnz), 256) + (most > back ? most : back);
}

// The step in one pass, if the call is one that small_step_kernel takes: its sizes, every operand present and aligned as
// the three passes require (which report what is not), no more label pairs than the workgroups' threads hold, and a
// workspace for the partial sums of all workgroups.  XFC_OK with *taken false otherwise.
static int small_step(const void* X, int64_t ldx, void* W, int64_t ldw, void* Mo, int64_t ldm, const int32_t* rowptr,
                      const int32_t* colidx, const int64_t* pos_x, const int64_t* pos_y, int64_t nnz, void* G, int64_t ldg,
                      float* dX, int64_t lddx, int64_t B, int64_t L, int64_t d, float lr, float momentum,
                      float weight_decay, float scale, void* ws, size_t ws_bytes, hipStream_t st, bool* taken) {
  *taken = false;
  if (B < 1 || B > SMALL_MAX_ROWS || !dims_ok(L) || L < 1 || !dims_ok(d) || nnz < 0 || nnz > SMALL_MAX_PAIRS) return XFC_OK;
  if (!X || !W || !Mo || !G || !dX || (nnz > 0 && !((rowptr && colidx) || (pos_x && pos_y)))) return XFC_OK;
  // With 33 to 64 rows of 768 dims the one pass fetches nothing ahead (see SmallStep::AHEAD), and each workgroup leaves 192 KB of
  // partial sums for a few tiles: G by itself and both gradients after it are faster while W and Mo stay in the caches, 64 rows x
  // 4,097 labels 32.6 -> 26.7 us, x 20,011 52.6 -> 44.4, but x 40,009 70 -> 74 and 33 rows x 40,009 61 -> 69.
  if (B > 32 && d >= 768 && L * d <= (int64_t)16 << 20) return XFC_OK;
  if (ldx % 8 || ldw % 8 || ldm % 8 || ldg % 8 || ldg < round_up(L, 8) || !aligned16(X) || !aligned16(W) || !aligned16(Mo) ||
      !aligned16(G) || !aligned16(ws))
    return XFC_OK;
  const size_t need = small_step_ws_bytes(B, L, d);
  if (need == 0 || ws_bytes < need) return XFC_OK;
  SmallArgs a = small_args(X, ldx, W, ldw, rowptr, colidx, pos_x, pos_y, nnz, G, ldg, B, L);
  a.Mo = (half_t*)Mo; a.ldm = ldm; a.lr = lr; a.mu = momentum; a.wd = weight_decay; a.part = reinterpret_cast<float*>(ws);
  int rc = XFC_OK;
  small_step_for(B, d, small_step_large(L, d), [&](auto s) {
    using S = decltype(s);
    const int grid = small_step_grid<S>(L);
    rc = launch_k<small_step_kernel<S>>(dim3((unsigned)grid), dim3(S::NT), S::LDS_BYTES, st, a);
    if (rc) return;
    launch_dx_reduce(a.part, dX, lddx, (int)B, (int)d, grid, scale, 0.0f, st);
    rc = check_launch();
  });
  *taken = true;
  return rc;
}

static int step_impl(const void* X, int64_t ldx, void* W, int64_t ldw, void* Mo, int64_t ldm, const int32_t* rowptr,
                     const int32_t* colidx, const int64_t* pos_x, const int64_t* pos_y, int64_t nnz, void* G, int64_t ldg,
                     float* dX, int64_t lddx, int64_t B, int64_t L, int64_t d, float lr, float momentum,
                     float weight_decay, float scale, void* workspace, size_t workspace_bytes, void* stream) {
  const size_t off = (size_t)round_up(xfc_fwd_grad_workspace_bytes(L, nnz), 256);
  if (!workspace || workspace_bytes < off) return XFC_ERR_WORKSPACE;  // xfc_dx checks its own share
  if (ldg < round_up(L, 8)) return XFC_ERR_SHAPE;
  unsigned char* ws = reinterpret_cast<unsigned char*>(workspace);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  bool taken;
  int rc = small_step(X, ldx, W, ldw, Mo, ldm, rowptr, colidx, pos_x, pos_y, nnz, G, ldg, dX, lddx, B, L, d, lr, momentum,
                      weight_decay, scale, ws + off, workspace_bytes - off, st, &taken);
  if (taken) return rc;
  rc = fwd_grad_impl(X, ldx, W, ldw, rowptr, colidx, pos_x, pos_y, nnz, G, ldg, B, L, d, nullptr, ws, off, st);
  if (rc) return rc;
  return xfc_dx_dw_update(G, ldg, X, ldx, W, ldw, Mo, ldm, dX, lddx, B, L, d, lr, momentum, weight_decay, scale, ws + off,
                          workspace_bytes - off, stream);
}

int xfc_step_csr(const void* X, int64_t ldx, void* W, int64_t ldw, void* Mo, int64_t ldm, const int32_t* rowptr,
                 const int32_t* colidx, int64_t nnz, void* G, int64_t ldg, float* dX, int64_t lddx, int64_t B,
                 int64_t L, int64_t d, float lr, float momentum, float weight_decay, float scale, void* workspace,
                 size_t workspace_bytes, void* stream) {
  if (B > 0 && !rowptr) return XFC_ERR_INVALID;
  return step_impl(X, ldx, W, ldw, Mo, ldm, rowptr, colidx, nullptr, nullptr, nnz, G, ldg, dX, lddx, B, L, d, lr, momentum,
                   weight_decay, scale, workspace, workspace_bytes, stream);
}

int xfc_step_coo(const void* X, int64_t ldx, void* W, int64_t ldw, void* Mo, int64_t ldm, const int64_t* pos_x,
                 const int64_t* pos_y, int64_t nnz, void* G, int64_t ldg, float* dX, int64_t lddx, int64_t B, int64_t L,
                 int64_t d, float lr, float momentum, float weight_decay, float scale, void* workspace,
                 size_t workspace_bytes, void* stream) {
  if (nnz > 0 && !(pos_x && pos_y)) return XFC_ERR_INVALID;
  return step_impl(X, ldx, W, ldw, Mo, ldm, nullptr, nullptr, pos_x, pos_y, nnz, G, ldg, dX, lddx, B, L, d, lr, momentum,
                   weight_decay, scale, workspace, workspace_bytes, stream);
}

// The K <= 8 pass.  Up to 32 rows whose fragments fit the LDS the weights stream past them (score_small_kernel), above that
// the forward pass's main loop runs (both sides of the line: score_wide_kernel); each leaves the largest score of every block.
// From some 400 MB of weights on, more than the caches hold, the main loop's whole lines are faster from the third row on: 32
// rows x 1,500,001 x 768 468 against 430 us, 16 x 2,300,001 x 512 467 against 443, 8 x 2,500,003 x 256 286 against 261; 1 row x
// 1,500,001 x 768 402 against 407.
constexpr int64_t SCORE_SMALL_BYTES = (int64_t)400 << 20;
struct TopkPlan {
  bool small;
  int block;          // labels per block
  int64_t range, ldb; // labels handled at a time, blocks of a row of the maxima (a multiple of 4)
};
static int64_t topk_blocks(int64_t labels, int block) { return round_up(ceil_div(labels, block), 4); }
// With a workspace that does not hold all maxima the labels go in ranges, the K best of each carried to the next.
static TopkPlan topk_plan(int64_t B, int64_t L, int64_t d, int64_t K, size_t ws_limit) {
  TopkPlan p;
  p.small = B <= SCORE_SMALL_ROWS && (B <= 2 || L * d * 2 <= SCORE_SMALL_BYTES) && (B <= 16 ? score_small_lds<1>(d) : score_small_lds<2>(d)) <= FULL_LDS;
  p.block = p.small ? SCORE_SMALL_BLOCK : SCORE_WIDE_BLOCK;
  p.range = L;
  // a tile of the wide kernel writes the maxima of all its blocks
  p.ldb = p.small ? topk_blocks(L, p.block) : topk_blocks(round_up(L, FwdWide::BM), p.block);
  if ((size_t)B * (size_t)p.ldb * 4 > ws_limit || L > TOPK_RANGE_MAX) {
    const int64_t lists = B * K * 8, unit = p.small ? 4 : FwdWide::BM / SCORE_WIDE_BLOCK, most = TOPK_RANGE_MAX / p.block;
    const int64_t fit = ws_limit > (size_t)lists ? (int64_t)((ws_limit - (size_t)lists) / ((size_t)B * 4)) : 0;
    p.ldb = (fit < most ? fit : most) / unit * unit;
    p.range = p.ldb * p.block;
  }
  return p;
}

constexpr int TOPK_SAMPLE = 2048;
// The pass with lists (topk_lists.hpp).  Label groups: enough to give every CU a workgroup, fewer when the workspace holds no
// more (8 at least; the seeding is dropped before the last groups are).  The rows' bounds start from the K-th score over a sample
// of the first TOPK_SAMPLE labels (a small logits pass and an exact selection) when every label group has enough tiles for that
// to pay; otherwise from nothing.  Without it every workgroup's first tiles overflow the candidate buffers and are rescanned.
struct ListPlan { int tiles_m, tiles_n, groups; bool seeded; size_t need; };
static ListPlan topk_list_plan(int64_t B, int64_t L, int64_t K, size_t ws_limit) {
  ListPlan p;
  p.tiles_m = ceil_div(B, row_tile(B));
  p.tiles_n = ceil_div(L, ListCore::BN);
  const int per = num_cus() / (8 * p.tiles_m);  // groups per XCD
  const int cap = (int)round_up(p.tiles_n, 8);
  p.groups = 8 * (per > 1 ? per : 1) < cap ? 8 * (per > 1 ? per : 1) : cap;
  for (;; p.groups -= 8) {
    // the groups' lists, the rows' shared bounds, and the sample's logits and their top K
    const size_t lists = (size_t)p.groups * B * K * 8 + (size_t)round_up(B, 4) * 4, sample = (size_t)B * TOPK_SAMPLE * 2 + (size_t)B * K * 12;
    p.seeded = L >= 8 * (int64_t)TOPK_SAMPLE && p.tiles_n >= 8 * p.groups && lists + sample <= ws_limit;
    p.need = lists + (p.seeded ? sample : 0);
    if (p.need <= ws_limit || p.groups <= 8) return p;
  }
}
// Lists or maxima.  A workspace that holds the maxima of a third of the labels or more takes those range by range (1024 rows x 131,072
// x 768, K = 5, three ranges 345 us, lists 386; 16 rows, four: 132 and 103); with less, launches and half-filled rounds add up (64
// rows x 131,072, K = 1, nine: 196 and 92; x 700,001, K = 5, ten: 377 and 247; what the least takes, see topk_lists.hpp).  Lists of
// more places cost the larger row tiles more: 65 to 512 rows with K from 4 on go up to nine ranges (128 rows x 700,001 x 64, nine: 155
// and 213; 512 x 131,072 x 768, eight: 651 and 712; ten: 128 x 700,001 x 768 387 and 359).  With room for all of them lists
// are the faster where storing and reading the maxima of very many labels weighs more than keeping lists of one to three places: up
// to 128 rows, K = 1 from some 1.25 million labels on (64 rows x 1,500,001 x 512 319 against 285 us, x 2,812,281 x 768 830 against 733;
// x 1,000,003 x 768 no difference), K = 2 and 3 from some 2 million on (64 x 2,812,281 x 768 1.12 and 1.08 times as fast, x 512 1.12
// and 1.06), at widths whose weights take their time either way (x 2,812,281 x 256, K = 3: 0.88); up to 3 rows of 768 dims for every
// K, where one workgroup a row reads all its maxima (1 row x 2,812,281 x 768, K = 5: 740 against 706 us).
static bool topk_by_lists(const TopkPlan& p, int64_t B, int64_t L, int64_t d, int64_t K) {
  if (L > TOPK_RANGE_MAX) return false;
  if (p.range < L) return (K >= 4 && B > 64 && B <= 512 ? 9 : 3) * p.range < L;
  if (B > 128 || d < 256) return false;
  if (K == 1) return L > 1250000;
  return L > 2000000 && d <= 768 && (K == 2 ? d >= 512 || B <= 64 : K == 3 ? d >= 512 : d > 512 && B <= 3);
}
// What the pass refuses to run without (lists of eight label groups), and what it runs fastest with.
static size_t topk_least(int64_t B, int64_t K) { return (size_t)8 * B * K * 8 + (size_t)round_up(B, 4) * 4; }
static size_t topk_need(int64_t B, int64_t L, int64_t K) {
  // whichever kernel the width leads to
  const size_t wide = (size_t)B * (size_t)topk_blocks(round_up(L, FwdWide::BM), SCORE_WIDE_BLOCK) * 4;
  const size_t small = B <= SCORE_SMALL_ROWS ? (size_t)B * (size_t)topk_blocks(L, SCORE_SMALL_BLOCK) * 4 : 0;
  const size_t need = wide > small ? wide : small, least = topk_least(B, K);
  return need > least ? need : least;
}

size_t xfc_topk_workspace_bytes(int64_t B, int64_t L, int64_t K) {
  if (!dims_ok(B) || !dims_ok(L) || K < 1 || K > SEL_MAX_K || B == 0 || L == 0) return 0;
  if (K > TOPK_MAX) return (size_t)B * (size_t)round_up(L, 8) * 2;  // the logits of every row
  return topk_need(B, L, K);
}

size_t xfc_layer_workspace_bytes(int64_t max_batch, int64_t L, int64_t d, int64_t max_nnz) {
  if (!dims_ok(max_batch) || !dims_ok(L) || !dims_ok(d) || max_nnz < 0) return 0;
  size_t dx = 0, topk = 0;
  const int64_t k8 = L < TOPK_MAX ? L : TOPK_MAX;
  for (int64_t b = 1; b <= max_batch; ++b) {
    const size_t a = xfc_dx_workspace_bytes(b, L, d), small = small_step_ws_bytes(b, L, d), back = back_ws_bytes(b, L, d);
    if (a > dx) dx = a;
    if (back > dx) dx = back;
    if (small > dx) dx = small;
    const size_t t = k8 > 0 ? xfc_topk_workspace_bytes(b, L, k8) : 0;
    if (t > topk) topk = t;
  }
  const size_t step = (size_t)round_up(xfc_fwd_grad_workspace_bytes(L, max_nnz), 256) + dx;
  return step > topk ? step : topk;
}

static int topk_lists(const half_t* X, int64_t ldx, const half_t* W, int64_t ldw, int B, int L, int d, int64_t numy, int K, float* values,
                      int64_t* indices, void* workspace, size_t workspace_bytes, hipStream_t st) {
  const ListPlan p = topk_list_plan(B, L, K, workspace_bytes);
  if (workspace_bytes < p.need) return XFC_ERR_WORKSPACE;
  ListArgs a;
  a.X = X; a.ldx = ldx; a.W = W; a.ldw = ldw;
  a.M = B; a.N = L; a.K = d; a.topk = K;
  a.tiles_m = p.tiles_m; a.tiles_n = p.tiles_n; a.n_groups = p.groups;
  a.cand_v = reinterpret_cast<float*>(workspace);
  a.cand_i = reinterpret_cast<int32_t*>(a.cand_v + (size_t)p.groups * B * K);
  a.bound = reinterpret_cast<uint32_t*>(a.cand_i + (size_t)p.groups * B * K);
  const dim3 rows((unsigned)ceil_div(B, 256));
  int rc;
  if (p.seeded) {
    // 16-byte aligned: the lists above are B * K * 8 * groups bytes (a multiple of 8 groups), the bounds 16-byte padded
    half_t* sample = reinterpret_cast<half_t*>(a.bound + round_up(B, 4));
    int64_t* sample_i = reinterpret_cast<int64_t*>(sample + (size_t)B * TOPK_SAMPLE);
    float* sample_v = reinterpret_cast<float*>(sample_i + (size_t)B * K);
    // by the list kernels' own loop, whatever the rows: topk_seed_kernel counts on sums that are theirs to the last bit
    const FwdPlan sums = {B <= 64 ? FWD_64 : FWD_128, TOPK_SAMPLE};
    rc = launch_fwd(sums, FWD_LINEAR, X, ldx, W, ldw, sample, TOPK_SAMPLE, B, TOPK_SAMPLE, d, TOPK_SAMPLE, 1.0f, 0.0f, st);
    if (rc) return rc;
    const SelArgs sa = {sample, (int64_t)TOPK_SAMPLE, TOPK_SAMPLE, (int64_t)TOPK_SAMPLE, K, 1, nullptr, 0, 0, sample_v, sample_i};
    if ((rc = launch_select<SEL_CAP_SMALL>(B, sa, st))) return rc;
    hipLaunchKernelGGL(topk_seed_kernel, rows, dim3(256), 0, st, (const float*)sample_v, K, a.bound, (int64_t)B);
  } else {
    // a kernel, not a memset: the call may be recorded into a graph
    hipLaunchKernelGGL(fill_u32_kernel, rows, dim3(256), 0, st, a.bound, 0u, (int64_t)B);
  }
  if ((rc = check_launch())) return rc;
  auto launch = [&](auto core) {
    using C = typename decltype(core)::type;
    return launch_k<topk_list_kernel<C>>(dim3((unsigned)(p.tiles_m * p.groups)), dim3(C::NT), TopkLds<C>::BYTES, st, a);
  };
  switch (row_tile(B)) {
    case 64: rc = launch(std::type_identity<ListCore64>{}); break;
    case 128: rc = launch(std::type_identity<ListCore128>{}); break;
    default: rc = launch(std::type_identity<ListCore>{}); break;
  }
  if (rc) return rc;
  hipLaunchKernelGGL(topk_merge_kernel, dim3((unsigned)B), dim3(256), 0, st, a.cand_v, a.cand_i, B, p.groups, K, numy, values, indices);
  return check_launch();
}

static int topk_impl(const void* X, int64_t ldx, const void* W, int64_t ldw, int64_t B, int64_t L, int64_t d, int64_t numy,
             int K, float* values, int64_t* indices, void* workspace, size_t workspace_bytes,
                     void* scratch, size_t scratch_bytes, void* stream) {
  if (!dims_ok(B) || !dims_ok(L) || !dims_ok(d)) return XFC_ERR_INVALID;
  if (B == 0) return XFC_OK;
  if (K < 1 || K > SEL_MAX_K || L < K || numy < 1 || d <= 0) return XFC_ERR_INVALID;
  if (!X || !W || !values || !indices) return XFC_ERR_INVALID;
  if (ldx % 8 || ldw % 8 || d % 8 || !aligned16(X) || !aligned16(W)) return XFC_ERR_ALIGN;
  if (K > TOPK_MAX) {
    // logits of a block of rows into the workspace, then an exact selection per row
    const int64_t ldl = round_up(L, 8);
    const int64_t fit = workspace ? (int64_t)(workspace_bytes / (size_t)(ldl * 2)) : 0;
    if (fit < (B < 256 ? B : 256)) return XFC_ERR_WORKSPACE;
    if (!aligned16(workspace)) return XFC_ERR_ALIGN;
    const int64_t block = fit >= B ? B : fit / 256 * 256;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // The blocks' maxima, if there is a place for them: the scratch, or what the logits leave of the workspace.  Rows of fewer
    // than 2048 blocks are read as fast without (1024 rows x 20,011, K = 100: 68 against 72 us; x 66,000: 120 against 87); from
    // two blocks per label sought on the bound leaves at most some 45 K candidates.
    const int64_t n_blocks = ceil_div(L, LOGIT_BLOCK), ldb = round_up(L, FwdWide::BM) / LOGIT_BLOCK;
    const size_t logits = (size_t)round_up((int64_t)((size_t)block * (size_t)ldl * 2), 16), maxima = (size_t)block * (size_t)ldb * 2;
    half_t* bmax = nullptr;
    if (K <= SEL_BLOCKS_MAX_K && n_blocks >= 2 * (int64_t)K && n_blocks >= SEL_BLOCKS_MIN) {
      if (scratch && scratch_bytes >= maxima && aligned16(scratch)) bmax = (half_t*)scratch;
      else if (workspace_bytes >= logits + maxima) bmax = (half_t*)((unsigned char*)workspace + logits);
    }
    for (int64_t r0 = 0; r0 < B; r0 += block) {
      const int64_t rows = B - r0 < block ? B - r0 : block;
      int rc = launch_fwd(fwd_plan(rows, L, d, false, num_cus()), FWD_LINEAR, (const half_t*)X + r0 * ldx, ldx, (const half_t*)W, ldw,
                          (half_t*)workspace, ldl, (int)rows, (int)L, (int)d, (int)L, 1.0f, 0.0f, st, NO_LOSS, bmax, ldb);
      if (rc) return rc;
      // sample every stride-th 16 KB block first when that still holds 16 K elements and points at about a
      // thousand candidates at most (half the sort buffer)
      const int cap = K <= SEL_SMALL_MAX_K ? SEL_CAP_SMALL : SEL_CAP_LARGE;
      int stride = 1;
      while (stride < 16 && (int64_t)K * stride * 2 <= cap / 2 && L / (stride * 2) >= 16 * (int64_t)K &&
             L / (stride * 2) >= (int64_t)SEL_THREADS * 8 * 4)
        stride *= 2;
      const SelArgs sa = {(const half_t*)workspace, ldl, (int)L, numy, K, stride, bmax, ldb, bmax ? (int)n_blocks : 0,
                          values + r0 * K, indices + r0 * K};
      rc = K <= SEL_SMALL_MAX_K ? launch_select<SEL_CAP_SMALL>((int)rows, sa, st) : launch_select<SEL_CAP_LARGE>((int)rows, sa, st);
      if (rc) return rc;
    }
    return XFC_OK;
  }
  if (!workspace || workspace_bytes < topk_least(B, K)) return XFC_ERR_WORKSPACE;
  if (!aligned16(workspace)) return XFC_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const TopkPlan p = topk_plan(B, L, d, K, workspace_bytes);
  if (topk_by_lists(p, B, L, d, K))
    return topk_lists((const half_t*)X, ldx, (const half_t*)W, ldw, (int)B, (int)L, (int)d, numy, K, values, indices, workspace,
                      workspace_bytes, st);
  if (p.range < 1) return XFC_ERR_WORKSPACE;
  for (int64_t l0 = 0; l0 < L; l0 += p.range) {
    const int64_t n = L - l0 < p.range ? L - l0 : p.range;
    ScoreArgs a;
    a.X = (const half_t*)X; a.ldx = ldx; a.W = (const half_t*)W + l0 * ldw; a.ldw = ldw;
    a.bmax = reinterpret_cast<float*>(workspace); a.ldb = p.ldb;
    a.M = (int)B; a.N = (int)n; a.K = (int)d;
    int rc;
    if (p.small) {
      rc = B <= 16 ? launch_score_small<1>(a, st) : launch_score_small<2>(a, st);
    } else {
      a.tiles_m = ceil_div(B, row_tile(B) <= 128 ? ScoreWide128::BN : ScoreWide::BN);
      a.tiles_n = ceil_div(n, ScoreWide::BM);
      const int64_t ids = (int64_t)a.tiles_m * round_up(a.tiles_n, 8);
      if (ids > 0x7fffffff) return XFC_ERR_INVALID;
      a.n_ids = (int)ids;
      auto launch = [&](auto core) {
        using C = typename decltype(core)::type;
        return launch_k<score_wide_kernel<C>>(dim3((unsigned)persistent_grid(ids, 1, num_cus())), dim3(C::NT), C::LDS_BYTES, st, a);
      };
      rc = row_tile(B) <= 128 ? launch(std::type_identity<ScoreWide128>{}) : launch(std::type_identity<ScoreWide>{});
    }
    if (rc) return rc;
    PickArgs k;
    k.X = a.X; k.ldx = ldx; k.W = a.W; k.ldw = ldw; k.bmax = a.bmax; k.ldb = p.ldb;
    k.n_blocks = ceil_div(n, p.block); k.N = (int)n; k.K = (int)d; k.first = l0; k.topk = K;
    k.best = p.range < L ? reinterpret_cast<unsigned long long*>(a.bmax + (size_t)B * p.ldb) : nullptr;
    k.begin = l0 == 0; k.end = l0 + n == L;
    k.numy = numy; k.out_v = values; k.out_i = indices;
    if (p.small) hipLaunchKernelGGL(topk_pick_kernel<SCORE_SMALL_BLOCK>, dim3((unsigned)B), dim3(512), 0, st, k);
    else hipLaunchKernelGGL(topk_pick_kernel<SCORE_WIDE_BLOCK>, dim3((unsigned)B), dim3(512), 0, st, k);
    if ((rc = check_launch())) return rc;
  }
  return XFC_OK;
}

int xfc_topk(const void* X, int64_t ldx, const void* W, int64_t ldw, int64_t B, int64_t L, int64_t d, int64_t numy,
             int K, float* values, int64_t* indices, void* workspace, size_t workspace_bytes, void* stream) {
  return topk_impl(X, ldx, W, ldw, B, L, d, numy, K, values, indices, workspace, workspace_bytes, nullptr, 0, stream);
}

int xfc_topk_scratch(const void* X, int64_t ldx, const void* W, int64_t ldw, int64_t B, int64_t L, int64_t d, int64_t numy,
                     int K, float* values, int64_t* indices, void* workspace, size_t workspace_bytes, void* scratch,
                     size_t scratch_bytes, void* stream) {
  return topk_impl(X, ldx, W, ldw, B, L, d, numy, K, values, indices, workspace, workspace_bytes, scratch, scratch_bytes, stream);
}

int xfc_copy(const void* src, void* dst, int64_t bytes, void* stream) {
  if (bytes < 0) return XFC_ERR_INVALID;
  if (bytes == 0) return XFC_OK;
  if (!src || !dst) return XFC_ERR_INVALID;
  if (bytes % 16 || !aligned16(src) || !aligned16(dst)) return XFC_ERR_ALIGN;
  const int64_t n16 = bytes / 16;
  int64_t grid = ceil_div(n16, 256);
  if (grid > 16384) grid = 16384;
  hipLaunchKernelGGL(copy_kernel, dim3((unsigned)grid), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     reinterpret_cast<const uint4v*>(src), reinterpret_cast<uint4v*>(dst), n16);
  return check_launch();
}

}  // extern "C"
