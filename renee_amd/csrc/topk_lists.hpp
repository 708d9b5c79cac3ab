// Top-K labels per row of X . W^T for K <= 8 with lists of the K best kept per workgroup, for workspaces that are short of the
// maxima that topk.hpp's kernels leave, and for few of the best out of very many labels.
//
// Each workgroup owns a row tile and walks every n_groups-th label tile with the forward main loop.  Per row it keeps the K best
// (score, label) pairs seen so far, ordered by score descending and label ascending (the order iterated torch.max produces: first
// maximum wins ties).  A finished tile is first filtered against each row's current K-th score; survivors (few once the lists have
// warmed up) go to a small per-row buffer that the row's owner thread merges.  If any row overflows its buffer, the tile is taken
// again exactly, a few columns at a time.  A second kernel merges the groups' lists.
// The workgroups that share a row tile also share what they have learnt: each publishes its rows' K-th scores to `bound` (atomic
// max) and filters against the largest published one as well.  Any published value is the K-th score of K real labels, so nothing
// below it can be in the row's final list; ties with it pass (a tying label of lower id may still rank above).  This only makes the
// filter tighter sooner: the lists, and so the results, do not depend on when a bound becomes visible.
//
// What bounds it, and where it is the faster: the lists take the LDS of the 256-row tile's third ring slot and a workgroup's first
// tiles are retaken, so that with room for the maxima topk.hpp's kernels win nearly everywhere (see topk_by_lists in xfc_kernels.hip).  But the
// workspace is 8 bytes per label group, row and place whatever the label count: 1024 rows x 2,812,281 x 768, K = 5, with 6.9 MB 4.34
// ms (the maxima, in 54 ranges of labels: 6.96), with 0.33 MB 25.8 (in 1,374 ranges: 98.7); 16 x 700,001 x 768, K = 1, 1,088 bytes
// 3.7 ms (in 3,647 ranges 60.9).
#pragma once
#include "pipe_core.hpp"
#include "topk.hpp"

namespace xfc {

constexpr int32_t TOPK_NO_LABEL = 0x7fffffff;
// Filtered candidates a row can take per tile on the fast path.  What the LDS leaves room for is 6; the 64-row tile has
// room for 32, a whole 32-column block, which turns the exact retake of a tile from 32 staged pieces of 8 columns into 8
// blocks of which only the candidates are looked at.  With small batches the label groups are one or two tiles long, so
// the first tile of each, which starts from no bound, is much of the work: 16 rows x 131,072 labels x 768, K = 5: the
// pass took 171 us with the staged retake on the 64-row tile, now 99.
using ListCore = PipeCore<256, 256, 64, 2, 4, 2, true, true, false, false, false, 4>;  // the lists take a third slot's LDS
using ListCore128 = PipeCore<128, 256, 64, 2, 4, 3, true, true, false, false, false, 4>;
using ListCore64 = PipeCore<64, 256, 64, 2, 4, 3, true, true, false, false, false, 4>;
template <class C>
constexpr int TOPK_CAP = C::BM == 64 ? 32 : 6;
template <class C>
struct TopkLds {
  float list_v[C::BM][TOPK_MAX];
  int32_t list_i[C::BM][TOPK_MAX];
  float tau[C::BM];
  int32_t cnt[C::BM];
  static constexpr int CAP = TOPK_CAP<C>;
  float buf_v[C::BM][CAP];  // candidates; CAP < 32, slow path: 8 staged columns (with buf_i)
  int32_t buf_i[C::BM][CAP];
  int32_t overflow;
  static constexpr int BYTES = C::LDS_BYTES + (int)(sizeof(float) * C::BM * (2 * TOPK_MAX + 2 + 2 * TOPK_CAP<C>) + 16);
};
static_assert(TopkLds<ListCore>::BYTES <= 160 * 1024 && TopkLds<ListCore128>::BYTES <= 160 * 1024 &&
              TopkLds<ListCore64>::BYTES <= 160 * 1024, "top-K LDS budget");
static_assert(2 * TOPK_CAP<ListCore> >= 8, "the exact rescan stages 8 columns in the candidate buffers");

struct ListArgs {
  const half_t* X; int64_t ldx;
  const half_t* W; int64_t ldw;
  int M, N, K;          // rows, labels, feature dims
  int topk;
  float* cand_v; int32_t* cand_i;  // [n_groups][M][topk]
  uint32_t* bound;                 // [M] shared lower bounds of the rows' final K-th scores (ordered keys, 0 = none yet)
  int tiles_m, tiles_n, n_groups;
};

// A value strictly below x (x finite or +inf) and as close to it as a normal number allows: "v > below(x)"
// admits every v >= x.  Tiny magnitudes step to a fixed small negative so that no denormal is ever compared.
__device__ __forceinline__ float topk_below(float x) {
  if (fabsf(x) < 1e-30f) return -1e-30f;
  const uint32_t b = __float_as_uint(x);
  return __uint_as_float(x > 0.f ? b - 1u : b + 1u);
}

__device__ __forceinline__ bool topk_better(float av, int ai, float bv, int bi) {
  return av > bv || (av == bv && ai < bi);
}
__device__ __forceinline__ void topk_insert(float* lv, int32_t* li, int K, float v, int i) {
  if (!topk_better(v, i, lv[K - 1], li[K - 1])) return;
  int p = K - 1;
  while (p > 0 && topk_better(v, i, lv[p - 1], li[p - 1])) {
    lv[p] = lv[p - 1];
    li[p] = li[p - 1];
    --p;
  }
  lv[p] = v;
  li[p] = i;
}

// The same on a list of TOPK_MAX held in registers.
__device__ __forceinline__ void topk_insert_regs(float (&lv)[TOPK_MAX], int32_t (&li)[TOPK_MAX], float v, int i) {
#pragma unroll
  for (int j = TOPK_MAX - 1; j >= 0; --j) {
    const bool here = topk_better(v, i, lv[j], li[j]);
    const bool above = j > 0 && topk_better(v, i, lv[j > 0 ? j - 1 : 0], li[j > 0 ? j - 1 : 0]);
    const float sv = above ? lv[j > 0 ? j - 1 : 0] : v;
    const int32_t si = above ? li[j > 0 ? j - 1 : 0] : i;
    lv[j] = here ? sv : lv[j];
    li[j] = here ? si : li[j];
  }
}

// Inlined on purpose: a function that is called waits for every outstanding memory operation on entry
// (the calling convention cannot know what is in flight), which here is the next tile's prefetch.
template <class S_t>
__device__ __forceinline__ void topk_push(S_t& S, int row, float v, int col) {
  const int slot = atomicAdd(&S.cnt[row], 1);
  if (slot < S_t::CAP) { S.buf_v[row][slot] = v; S.buf_i[row][slot] = col; }
  else S.overflow = 1;
}

template <class C>
__global__ void __launch_bounds__(C::NT) topk_list_kernel(ListArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
  half_t* lds = reinterpret_cast<half_t*>(smem_raw);
  TopkLds<C>& S = *reinterpret_cast<TopkLds<C>*>(smem_raw + C::LDS_BYTES);
  // ids are dealt round-robin to XCDs: the row tiles of one label group sit side by side on one XCD
  const int mt = (blockIdx.x >> 3) % a.tiles_m, grp = (blockIdx.x >> 3) / a.tiles_m * 8 + (blockIdx.x & 7);
  const int n_items = grp < a.tiles_n ? (a.tiles_n - grp + a.n_groups - 1) / a.n_groups : 0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int m0 = mt * C::BM;
  const int K = a.topk;
  // What the filter compares with, tau: a score at or below it stays out.  A list that is not full takes scores of -inf too: with
  // NONE nothing stays out, and scores that are no number are dropped behind the filter.  Where a tile can be retaken by whole
  // blocks it is, as long as a row has neither a bound nor a full list, and the filter need not know of NONE.
  constexpr bool BLOCKS = TopkLds<C>::CAP >= 32;
  const float NEG_INF = -__builtin_huge_valf(), NONE = BLOCKS ? NEG_INF : __builtin_nanf("");
  auto passes = [](float v, float tau) { return BLOCKS ? v > tau : !(v <= tau); };
  auto bound_of = [&](uint32_t key) { return key > topk_key(NEG_INF) ? topk_below(topk_unkey(key)) : NONE; };
  if (threadIdx.x == 0) S.overflow = 0;
  __syncthreads();
  for (int t = threadIdx.x; t < C::BM; t += C::NT) {
    for (int j = 0; j < TOPK_MAX; ++j) { S.list_v[t][j] = NEG_INF; S.list_i[t][j] = TOPK_NO_LABEL; }
    // the first tile is filtered against a seeded bound, if there is one (1024 rows x 2,812,281 labels: 4.54 -> 4.32 ms
    // against a first tile that starts from nothing and is taken twice); rows past the batch never take anything
    float tau = -NEG_INF;
    if (m0 + t < a.M) tau = bound_of(__hip_atomic_load(a.bound + m0 + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    S.tau[t] = tau;
    S.cnt[t] = 0;
    // without one the first tile is taken the exact way at once
    if (BLOCKS && tau == NONE) S.overflow = 1;
  }
  __syncthreads();

  auto get = [&](int item, typename C::Operand& oa, typename C::Operand& ob, int& kb, int& ke) {
    const int nt = grp + item * a.n_groups;
    oa = typename C::Operand{a.X, a.ldx, m0, a.M, a.K};
    ob = typename C::Operand{a.W, a.ldw, nt * C::BN, a.N, a.K};
    kb = 0;
    ke = a.K;
  };
  auto epilogue = [&](int item, float16v (&acc)[C::FM][C::FN]) {
    const int nt = grp + item * a.n_groups;
    const int n0 = nt * C::BN;
    const bool ragged = n0 + C::BN > a.N;
    const int h = lane >> 5;
    // the row owners ask for the shared bound now and use it after the filter
    const bool owner = threadIdx.x < C::BM && m0 + (int)threadIdx.x < a.M;
    uint32_t shared_key = 0u;
    if (owner) shared_key = __hip_atomic_load(a.bound + m0 + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // tau from the next tile on: the list's K-th score, or just below the shared bound
    auto settle = [&](int t, bool changed, bool retaken) {
      const float mine = S.list_i[t][K - 1] != TOPK_NO_LABEL ? S.list_v[t][K - 1] : NONE;
      if (changed && owner && mine > NEG_INF)
        __hip_atomic_fetch_max(a.bound + m0 + t, topk_key(mine), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const float bound = bound_of(shared_key);
      S.tau[t] = owner ? fmaxf(mine, bound) : -NEG_INF;  // (the one that is a number)
      // (the flag is only set where no wave still reads it, and a row that needs it has come through here)
      if (BLOCKS && retaken && owner && bound == NONE && S.list_i[t][K - 1] == TOPK_NO_LABEL) S.overflow = 1;
      S.cnt[t] = 0;
    };
    // filter against each row's K-th best so far (a flag that is set already is the first tile's: wave-uniform, all agree)
    if (!BLOCKS || S.overflow == 0)
#pragma unroll
    for (int fm = 0; fm < C::FM; ++fm) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row0 = wm * C::TM + fm * 32 + 8 * q + 4 * h;
        const float4v tau4 = *reinterpret_cast<const float4v*>(&S.tau[row0]);
        // one branch per strip of 4 rows x TN labels: the compares are combined as lane masks, and only a
        // strip in which some lane holds a survivor walks its elements (rare once the lists have warmed up)
        bool any = false;
#pragma unroll
        for (int fn = 0; fn < C::FN; ++fn)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) any |= passes(acc[fm][fn][4 * q + rr], tau4[rr]);
        if (__builtin_amdgcn_ballot_w64(any) != 0) {
          // opaque on purpose: the compiler otherwise computes the list addresses of all 128 elements when
          // the kernel starts, spills them, and reloads them here behind a wait for every outstanding fetch
          int r0 = row0;
          asm volatile("" : "+v"(r0));
#pragma unroll
          for (int fn = 0; fn < C::FN; ++fn) {
            const int col = n0 + wn * C::TN + fn * 32 + (lane & 31);
            const bool col_ok = !ragged || col < a.N;
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
              const float v = acc[fm][fn][4 * q + rr];
              if (passes(v, tau4[rr]) && (BLOCKS || v == v) && col_ok) topk_push(S, r0 + rr, v, col);
            }
          }
        }
        asm volatile("" ::: "memory");  // keep the threshold reads of later strips from being hoisted up here
      }
    }
    __syncthreads();
    const bool overflow = S.overflow != 0;
    if (!overflow) {
      if (threadIdx.x < C::BM) {
        const int t = threadIdx.x;
        const int n = S.cnt[t];
        for (int i = 0; i < n; ++i) topk_insert(S.list_v[t], S.list_i[t], K, S.buf_v[t][i], S.buf_i[t][i]);
        settle(t, n != 0, false);
      }
    } else if constexpr (BLOCKS) {
      // exact retake, a block of 32 columns at a time: no row can have more candidates than its buffer holds, and from
      // the second block on only those that pass the bound the earlier blocks have raised ("at least tau" here).
      const int t = threadIdx.x;
      float lv[TOPK_MAX];
      int32_t li[TOPK_MAX];
      __syncthreads();
      if (t < C::BM) {
#pragma unroll
        for (int j = 0; j < TOPK_MAX; ++j) { lv[j] = S.list_v[t][j]; li[j] = S.list_i[t][j]; }
        S.cnt[t] = 0;
      }
      if (t == 0) S.overflow = 0;
      __syncthreads();
#pragma unroll
      for (int sfn = 0; sfn < C::FN; ++sfn) {
        for (int swn = 0; swn < C::WN; ++swn) {
          if (wn == swn) {
            const int col = n0 + swn * C::TN + sfn * 32 + (lane & 31);
            if (col < a.N) {
#pragma unroll
              for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                  const int row = wm * C::TM + fm * 32 + c_row(r, lane);
                  const float v = acc[fm][sfn][r];
                  if (v >= S.tau[row]) topk_push(S, row, v, col);
                }
            }
          }
          __syncthreads();
          if (t < C::BM) {
            const int n = S.cnt[t];
            for (int i = 0; i < n; ++i) topk_insert_regs(lv, li, S.buf_v[t][i], S.buf_i[t][i]);
            float kth = lv[0];
#pragma unroll
            for (int j = 1; j < TOPK_MAX; ++j) kth = j < K ? lv[j] : kth;
            S.tau[t] = fmaxf(S.tau[t], kth);
            S.cnt[t] = 0;
          }
          __syncthreads();
        }
      }
      if (t < C::BM) {
#pragma unroll
        for (int j = 0; j < TOPK_MAX; ++j) { S.list_v[t][j] = lv[j]; S.list_i[t][j] = li[j]; }
        settle(t, true, true);
      }
    } else {
      // exact rescan: stage 8 columns of all 256 rows at a time, each row's owner inserts them
      float* stage = &S.buf_v[0][0];  // 256 x 8 floats: buf_v and buf_i are adjacent
      __syncthreads();
#pragma unroll
      for (int swn = 0; swn < C::WN; ++swn) {
#pragma unroll
        for (int sfn = 0; sfn < C::FN; ++sfn) {
          for (int sg = 0; sg < 4; ++sg) {
            if (wn == swn && ((lane & 31) >> 3) == sg) {
#pragma unroll
              for (int fm = 0; fm < C::FM; ++fm)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                  stage[(wm * C::TM + fm * 32 + c_row(r, lane)) * 8 + (lane & 7)] = acc[fm][sfn][r];
            }
            __syncthreads();
            if (threadIdx.x < C::BM) {
              const int t = threadIdx.x;
              const int cbase = n0 + swn * C::TN + sfn * 32 + sg * 8;
              for (int e = 0; e < 8; ++e)
                if (cbase + e < a.N) topk_insert(S.list_v[t], S.list_i[t], K, stage[t * 8 + e], cbase + e);
            }
            __syncthreads();
          }
        }
      }
      if (threadIdx.x < C::BM) settle(threadIdx.x, true, true);
      if (threadIdx.x == 0) S.overflow = 0;
    }
    __syncthreads();
  };
  C::run(0, n_items, lds, get, epilogue);
  __syncthreads();
  if (threadIdx.x < C::BM && m0 + threadIdx.x < a.M && grp < a.n_groups) {
    const int64_t o = ((int64_t)grp * a.M + m0 + threadIdx.x) * K;
    for (int j = 0; j < K; ++j) { a.cand_v[o + j] = S.list_v[threadIdx.x][j]; a.cand_i[o + j] = S.list_i[threadIdx.x][j]; }
  }
}

// One workgroup per row, one thread per group (and every 256th): K rounds of "best head of the groups' lists", which are
// in order.  Bound by latency: the candidates are read once, up front.  (One wave per row that read all candidates anew in
// each round took 33 us for 256 groups, K = 5; this one 6.7.)
__global__ void __launch_bounds__(256) topk_merge_kernel(const float* __restrict__ cand_v, const int32_t* __restrict__ cand_i,
                                                         int M, int n_groups, int K, int64_t numy,
                                                         float* __restrict__ out_v, int64_t* __restrict__ out_i) {
  __shared__ unsigned long long wave_best[2][4];
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // this thread's best TOPK_MAX, in order; entries past K are those of a list that is not full, and lose to all others
  float lv[TOPK_MAX];
  int32_t li[TOPK_MAX];
#pragma unroll
  for (int j = 0; j < TOPK_MAX; ++j) { lv[j] = -__builtin_huge_valf(); li[j] = TOPK_NO_LABEL; }
  for (int g = threadIdx.x; g < n_groups; g += 256) {
    const int64_t o = ((int64_t)g * M + row) * K;
    if (g == (int)threadIdx.x) {
#pragma unroll
      for (int j = 0; j < TOPK_MAX; ++j)
        if (j < K) { lv[j] = cand_v[o + j]; li[j] = cand_i[o + j]; }
    } else {
      for (int j = 0; j < K; ++j) topk_insert_regs(lv, li, cand_v[o + j], cand_i[o + j]);
    }
  }
  for (int r = 0; r < K; ++r) {
    // score descending, then label ascending, as one number; a score of -0 ranks with +0
    const unsigned long long mine = ((unsigned long long)topk_key(lv[0] == 0.f ? 0.f : lv[0]) << 32) | (uint32_t)~li[0];
    unsigned long long best = mine;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned long long other = __shfl_xor(best, off, 64);
      best = other > best ? other : best;
    }
    if (lane == 0) wave_best[r & 1][wave] = best;
    __syncthreads();  // one per round: the next round writes the other half, and the one after it waits for this read
    best = wave_best[r & 1][0];
#pragma unroll
    for (int w = 1; w < 4; ++w) best = wave_best[r & 1][w] > best ? wave_best[r & 1][w] : best;
    if (mine == best) {  // one thread, or all that hold nothing more
      out_v[(int64_t)row * K + r] = lv[0];
      int64_t idx = li[0];
      if (idx >= numy) idx = numy - 1;  // padded labels are clamped, as the reference does, and places without a label
      out_i[(int64_t)row * K + r] = idx;
#pragma unroll
      for (int j = 0; j + 1 < TOPK_MAX; ++j) { lv[j] = lv[j + 1]; li[j] = li[j + 1]; }
      lv[TOPK_MAX - 1] = -__builtin_huge_valf();
      li[TOPK_MAX - 1] = TOPK_NO_LABEL;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// top-K for 8 < K <= 8192: exact selection over rows of fp16 logits (one workgroup per row)

// bound[r] = key of a value safely below the K-th largest of row r's sample scores.  The sample scores
// are fp16 roundings (half an ulp from the fp32 score at most) of sums made as the list kernels make them, the same MFMAs in
// the same order, so one part in 1024 plus the smallest fp16 step below the K-th rounded score is below the K-th fp32 score of the
// sample, hence of the whole row.  (Sums in another order differ by what they round off, relative to the products' magnitudes: where
// these cancel, by more than that.  The wide loop's 16x16x32 MFMAs happen to give the same bits: 211,000 best scores of operands over up
// to 21 binary orders of magnitude and of cancelling products.)
__global__ void __launch_bounds__(256) topk_seed_kernel(const float* __restrict__ sample_v, int K, uint32_t* __restrict__ bound,
                                                        int64_t n) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= n) return;
  const float first = sample_v[r * K], x = sample_v[r * K + K - 1];  // (a score that is no number ranks first there)
  const float lo = x - (fabsf(x) * 0.0009765625f + 1.2e-7f);
  bound[r] = first == first && lo == lo && lo > -__builtin_huge_valf() ? topk_key(lo) : 0u;  // 0: no bound
}

__global__ void __launch_bounds__(256) fill_u32_kernel(uint32_t* __restrict__ dst, uint32_t value, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = value;
}

}  // namespace xfc
