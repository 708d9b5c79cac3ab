// The main loop of pipe_core.hpp for the two large contractions (forward pass and dX on batches above 128 rows):
// four waves of 128 x 128 instead of eight of 128 x 64, 16x16x32 MFMAs, every LDS read and every fetch placed between
// two MFMAs, and a third ring slot for the operand that comes from HBM.
//
// Operands, swizzled LDS images and the meaning of KC and MC are those of pipe_core.hpp.
//
// MFMA 16x16x32 register layout (checked on hardware):
//   A: lane l holds A[i = l%16][k = 8*(l/16) .. +7]
//   B: lane l holds B[k = 8*(l/16) .. +7][j = l%16]
//   C: lane l, register r holds C[i = 4*(l/16) + r][j = l%16]
// so a lane's registers run along the A side's index: the kernels put on the A side whichever index is
// contiguous in the output.  A KC A side is stored in the LDS with its rows permuted inside every 32
// (LDS row 16b + 4g + r holds row 8g + 4b + r), which makes the two blocks of a 32-row pair give a lane eight
// consecutive rows: 16 bytes of fp16 output with no pass through the LDS.
//
// What bounds it.  A SIMD's matrix pipe takes 16 cycles for such an MFMA and 4 to issue it; with one wave per SIMD the
// pipe stays busy as long as no more than three other instructions stand between two MFMAs.  Counters at 512 x 1,310,720
// x 768 put dX at 2048 MFMA cycles of 2850 per stage (PipeCore: of 3100), the rest being the stage barrier and issue
// slots of the fetches (address and M0 arithmetic included).  The other
// bound is power: with random operands the chip lowers its clock (1.6 to 1.9 GHz here) the more the busier the pipes and
// the HBM are, so fewer LDS bytes and fewer stalled cycles count twice.  Measured on one card, back to back:
//   forward pass 1.21 -> 1.11 ms, dX 1.046 -> 0.926 ms (batch 512, 1,310,720 labels, d = 768) against PipeCore;
//   branches around fetches between MFMAs cost 15 % of a product that runs from the L2, fetch addresses made of a base and
//   two offsets (five scalar instructions a fetch) 6 % of dX, the third slot for the operand from HBM 9 % of the forward
//   pass (1.31 -> 1.19 ms), a fill cursor with a byte of state per slot 4 % of both.
// Then: what a stage does once (the turns of the rings, counts, the bumps, which the compiler had moved there) out of the gap
// between the sub-steps and behind their last bumps, tile to tile addresses by one difference, and an epilogue's stores counted
// instead of waited for: forward pass 1.055 -> 1.030 ms, dX 0.880 -> 0.865, the logits of top-100 at 512 x 1,310,720 1.113 ->
// 1.083 (top-5 of 1024 x 2,812,281 3.70 and 3.65 ms, no more than its runs differ by).
// Eight waves of 128 x 64 run no faster (1359 against 1360 TFLOP/s at 8192^3), read half again as many LDS bytes, and
// leave 128 registers for everything that is not an accumulator.
#pragma once
#include <type_traits>

#include "pipe_core.hpp"

namespace xfc {

// address = uniform 64-bit base + per-lane 32-bit offset; LDS address = uniform lds + the constant at
// SPILLED: the base may have been in a vector register's lane (scalar registers are spilled there).  Five instructions must stand
// between the v_readlane_b32 that brings it back and a vector-memory instruction that reads it, and the compiler does not see that
// there is one in the asm; a scalar move waits by itself, so the base goes through one.  (It stands where M0 wants one instruction
// before the fetch anyway, but the two registers cost the 1024-row top-K pass, which spills none of them, 1.2 %.  tests/test_host.py
// looks the built kernels over.)
template <bool NT = false, bool SPILLED = false>
__device__ __forceinline__ void wide_load16(int64_t ubase, uint32_t voff, uint32_t lds, int at) {
  // an integer operand whose halves are marked uniform: the "s" constraint alone is not always honoured
  const uint64_t b0 = (uint64_t)ubase;
  // (readfirstlane returns a signed int: widen through uint32_t, or the low half sign-extends into the high one)
  const uint32_t b_hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b0 >> 32));
  const uint32_t b_lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b0);
  const uint64_t b = ((uint64_t)b_hi << 32) | (uint64_t)b_lo;
  const uint32_t m = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds);
  if constexpr (SPILLED) {
    uint64_t t;
    if constexpr (NT)
      asm volatile("s_add_u32 m0, %1, %4\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0 nt" : "=&s"(t) : "s"(m), "v"(voff), "s"(b), "n"(at) : "memory", "m0", "scc");
    else
      asm volatile("s_add_u32 m0, %1, %4\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0" : "=&s"(t) : "s"(m), "v"(voff), "s"(b), "n"(at) : "memory", "m0", "scc");
  } else if constexpr (NT) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(m), "v"(voff), "s"(b), "n"(at) : "memory", "m0", "scc");
  } else {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m), "v"(voff), "s"(b), "n"(at) : "memory", "m0", "scc");
  }
}

// Swizzles: the 16 lanes (b128) or 32 lanes (b64) the LDS serves at a time must spread over all 64 banks.
// KC, 128-byte rows: the 16 rows of a fragment cover the 256 bytes of a bank line.
__device__ __forceinline__ int wide_kc_swz(int row) { return (row >> 1) & 7; }
// MC: half a wave reads 32 bytes of each of the k-rows {0..3, 8..11} (mod 16) of one column block; a k-row is 2R
// bytes with R a multiple of 128, so all eight rows start at the same bank and need eight different 32-byte segments.
__device__ __forceinline__ int wide_mc_swz(int k) { return ((k & 3) << 1) | (((k >> 3) & 1) << 3); }

// The A side comes from HBM: its ring has three slots, and it is fetched half a stage earlier than the B side, whose
// ring has two.  The B side is K-contiguous.
// SPILLED_: some of the fetches' addresses are spilled (see wide_load16).
template <int BM_, int BN_, int WM_, int WN_, bool A_KC_, bool SPILLED_ = false>
struct WideCore {
  static constexpr int BM = BM_, BN = BN_, BK = 64, WM = WM_, WN = WN_;
  static constexpr bool A_KC = A_KC_, SPILLED = SPILLED_;
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int TM = BM / WM, TN = BN / WN;   // a wave's tile
  static constexpr int FM = TM / 16, FN = TN / 16;   // in 16 x 16 blocks
  static constexpr int A_HALVES = BM * BK, B_HALVES = BN * BK;
  static constexpr int A_SLOTS = 3, B_SLOTS = 2;
  static constexpr int LDS_BYTES = (A_SLOTS * A_HALVES + B_SLOTS * B_HALVES) * 2;
  static constexpr int A_CH = BM * BK / 8 / NT, B_CH = BN * BK / 8 / NT;  // fetch instructions per wave and stage
  static constexpr int NM = FM * FN;                   // MFMAs of a sub-step of 32 k
  static constexpr int A_RD = A_KC ? FM : 2 * FM, B_RD = FN, NR = A_RD + B_RD;  // its fragment reads
  // A sub-step's reads go into the first half of the previous sub-step's MFMAs, so that the last has landed before it is
  // wanted.  The fetches that have less time to land (the B side's) go into the first half of the second sub-step,
  // the others are spread over the first.  A fetch's address is advanced two MFMAs after the next fetch.
  static constexpr int READ_EVERY = NM / (2 * NR) > 0 ? NM / (2 * NR) : 1;
  static constexpr int B_EVERY = NM / (2 * B_CH), A_EVERY = NM / (A_CH + 1);
  static_assert(BM % (32 * WM) == 0 && BN % (16 * WN) == 0, "wave tile: pairs of 16-row blocks by 16-column blocks");
  static_assert((BM * BK / 8) % NT == 0 && (BN * BK / 8) % NT == 0, "chunk split");
  static_assert(A_KC ? BM % 64 == 0 : BM % 128 == 0 && 512 % BM == 0, "swizzle; a fetch instruction covers whole k-rows");
  static_assert(BN % 64 == 0, "swizzle");
  static_assert((NR - 1) * READ_EVERY < NM, "the reads fit their sub-step");
  static_assert(B_EVERY > 1 && A_EVERY > 1 && B_CH * B_EVERY + 1 < NM && A_CH * A_EVERY + 1 < NM, "so do the fetches");
  static_assert(NW % 2 == 0, "the KC swizzle assumes that a fetch instruction's rows are 8 times an even step apart");

  // One operand's tile: base pointer, leading dimension (halves), first row (KC) or column (MC) of the tile and the limit
  // of that index.  Requirements: r0 < rmax; ld is a multiple of 8 and ld * 2 * 32 < 2^32; for MC operands rmax is a
  // multiple of 8.  Rows (columns) at or past rmax are fetched from the last valid row (column chunk) instead: they only
  // ever feed outputs the caller discards.  The limit of the contraction index is the item's k_end, up to which (KC: up to
  // the next multiple of 8) both operands must be readable: nothing past it is read, and what a stage holds past it counts
  // as zeros.
  struct Operand {
    const half_t* p;
    int64_t ld;
    int r0, rmax;
  };

  // A uniform value that is to be made here and not where it is used.
  __device__ __forceinline__ static void pin(int& v) {
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
  }
  __device__ __forceinline__ static void pin(uint32_t& v) {
    v = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    asm volatile("" : "+s"(v));
  }
  __device__ __forceinline__ static void pin(int64_t& v) {
    v = uniform64(v);
    asm volatile("" : "+s"(v));
  }
  // Addresses of the CH 16-byte pieces a thread fetches for one operand each stage.  Every fetch is
  // "uniform 64-bit address + per-thread 32-bit offset": the base advances along k with scalar adds, so a
  // steady-state stage costs no vector ALU work.
  template <bool KC, int R, int CH, bool PERM>
  struct Loader {
    static constexpr int CPI = KC ? BK / 8 : R / 8;  // 16-byte chunks per tile row (KC) or per k-row (MC)
    static constexpr int RPI = 64 / CPI;             // rows per instruction
    int64_t at[CH];      // uniform address of each instruction's first row at its next stage's first k
    int64_t kstep;       // uniform
    uint32_t voff[CH];   // per-thread byte offset from there
    __device__ __forceinline__ void init(const Operand& o, int k_begin, int wave, int lane) {
      if constexpr (KC) {
        const int sub = lane / CPI, pc = lane % CPI;
        const half_t* base = o.p + (int64_t)o.r0 * o.ld + k_begin;
        kstep = (int64_t)BK * 2;
        const int c = pc ^ wide_kc_swz(wave * RPI + sub);  // the swizzle does not depend on i (NW is even)
        const int last = o.rmax - 1 - o.r0;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          const int rho = (i * NW + wave) * RPI;  // first LDS row of the instruction
          // PERM: LDS row 16b + 4g + r <- row 8g + 4b + r of every 32 (see the head of the file)
          const int first = PERM ? (rho & ~31) + 8 * ((rho >> 2) & 3) + 4 * ((rho >> 4) & 1) : rho;
          const int rel = PERM ? 8 * (sub >> 2) + (sub & 3) : sub;
          const int g = first < last ? first : last;
          const int row = first + rel < last ? first + rel : last;
          at[i] = uniform64(reinterpret_cast<int64_t>(base + (int64_t)g * o.ld));
          voff[i] = (uint32_t)(row - g) * (uint32_t)(o.ld * 2) + (uint32_t)c * 16u;
        }
      } else {
        const half_t* base = o.p + (int64_t)k_begin * o.ld + o.r0;
        kstep = uniform64((int64_t)BK * o.ld * 2);
        const int last = o.rmax - 8 - o.r0;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          const int q = (i * NW + wave) * 64 + lane, k = q / CPI, pc = q % CPI;
          const int c = (pc ^ wide_mc_swz(k)) * 8;
          const int k0 = (i * NW + wave) * RPI;
          at[i] = uniform64(reinterpret_cast<int64_t>(base + (int64_t)k0 * o.ld));
          voff[i] = (uint32_t)(k - k0) * (uint32_t)(o.ld * 2) + (uint32_t)(c < last ? c : last) * 2u;
        }
      }
    }
    // For the stage that crosses k_end (n < BK of its k are left), the last of an item: lanes whose piece lies past the
    // end fetch an earlier k, which is inside the operand; clear_tail() replaces what they brought.
    __device__ __forceinline__ void retarget(int n, int64_t ld, int wave, int lane) {
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int k = piece_k(i, wave, lane);
        if constexpr (KC) {
          voff[i] -= k >= n ? (uint32_t)k * 2u : 0u;
        } else {
          const int k0 = (i * NW + wave) * RPI;  // the instruction's first k-row
          voff[i] -= k >= n ? (uint32_t)(k - k0) * (uint32_t)(ld * 2) : 0u;
          at[i] -= k0 < n ? 0 : uniform64((int64_t)k0 * ld * 2);
        }
      }
    }
    __device__ __forceinline__ static int piece_k(int i, int wave, int lane) {  // k of a piece inside its stage
      if constexpr (KC) return ((lane % CPI) ^ wide_kc_swz(wave * RPI + lane / CPI)) * 8;
      else return ((i * NW + wave) * 64 + lane) / CPI;
    }
    __device__ __forceinline__ static void clear_tail(half_t* region, int n, int wave, int lane) {
#pragma unroll
      for (int i = 0; i < CH; ++i)
        if (piece_k(i, wave, lane) >= n) *reinterpret_cast<uint4v*>(region + (i * NW + wave) * 512 + lane * 8) = uint4v{0u, 0u, 0u, 0u};
    }
    __device__ __forceinline__ void issue(int i, uint32_t wave_region) const { wide_load16<false, SPILLED>(at[i], voff[i], wave_region, i * NW * 1024); }
    __device__ __forceinline__ void bump(int i) {
      at[i] += kstep;
      pin(at[i]);
    }
  };
  // A fill cursor: the stage of the work list an operand's next fetches belong to.
  template <bool IS_A>
  struct Cursor {
    static constexpr int SLOTS = IS_A ? A_SLOTS : B_SLOTS, BYTES = (IS_A ? A_HALVES : B_HALVES) * 2, CH = IS_A ? A_CH : B_CH;
    using Load = std::conditional_t<IS_A, Loader<A_KC, BM, A_CH, A_KC>, Loader<true, BN, B_CH, false>>;
    Load load;
    uint32_t ring, dst;  // LDS address of this wave's first piece in slot 0 and in the stage's slot
    int item, k_left;    // k of the item from this stage on
    int64_t ld;
    int64_t shift;        // of the first address from where the item's tile starts
    bool inside = false;  // the tile lies inside the operand, its k are whole stages, and shift is known
    // MOVE: from one tile that lies inside the operand to another all addresses move by the same (made anew they are 150
    // instructions between two stages).  Not from the first one: what that takes would stand in front of every kernel's first
    // stage, 0.3 us of a small one's 20.
    template <bool MOVE, class GetItem>
    __device__ __forceinline__ void open(GetItem& get, int wave, int lane) {
      Operand o[2];
      int kb, ke;
      get(item, o[0], o[1], kb, ke);
      const Operand& me = o[IS_A ? 0 : 1];
      if constexpr (MOVE) {
        constexpr bool KC = IS_A ? A_KC : true;
        const bool was = inside;
        inside = me.r0 + (IS_A ? BM : BN) <= me.rmax && (ke - kb) % BK == 0;
        const int64_t start = uniform64(reinterpret_cast<int64_t>(me.p) + (KC ? me.r0 * me.ld + kb : kb * me.ld + me.r0) * 2);
        if (was && inside) {
          const int64_t by = uniform64(start + shift - load.at[0]);
#pragma unroll
          for (int i = 0; i < CH; ++i) load.at[i] += by;
        } else {
          load.init(me, kb, wave, lane);
          shift = uniform64(load.at[0] - start);
        }
      } else {
        load.init(me, kb, wave, lane);
      }
      ld = me.ld;
      k_left = ke - kb;
      if (k_left < BK) load.retarget(k_left, ld, wave, lane);
    }
    __device__ __forceinline__ void piece(int i) const { load.issue(i, dst); }
    __device__ __forceinline__ void bump(int i) { load.bump(i); }
    // To the next stage, whose addresses bump() has made: what every stage has, for a place among the MFMAs (and pinned there), and
    // what the end of an item needs.  Past the last one the cursor stays: later fetches repeat it, nobody reads the copies, and
    // the count of outstanding fetches per stage stays what the waits assume.
    __device__ __forceinline__ void step() {
      dst = dst == ring + (SLOTS - 1) * BYTES ? ring : dst + BYTES;
      k_left -= BK;
      pin(dst);
      pin(k_left);
    }
    template <bool MOVE, class GetItem>
    __device__ __forceinline__ void turn(GetItem& get, int item_end, int wave, int lane) {
      if (k_left < BK) {
        if (k_left > 0) {
          load.retarget(k_left, ld, wave, lane);
        } else if (item + 1 < item_end) {
          ++item;
          open<MOVE>(get, wave, lane);
        } else {
          k_left += BK;
#pragma unroll
          for (int i = 0; i < CH; ++i) load.at[i] -= load.kstep;
        }
      }
    }
  };

  struct Frags {
    half8 a[FM], b[FN];
  };
  // One LDS read of a fragment: KC, the whole 16 x 32 block (rows r0 ..); MC, half of the k of the block whose columns
  // start at r0 (within each 16-lane group, lane t supplies the address of row k + t/4, columns r0 + 4*(t%4)..+3 and
  // receives column r0 + t for four consecutive k).
  template <bool KC, int R>
  __device__ __forceinline__ static void read_piece(const half_t* lds, int r0, int kk, int half, int lane, half8& f) {
    if constexpr (KC) {
      const int r = r0 + (lane & 15), c = kk * 4 + (lane >> 4);
      f = *reinterpret_cast<const half8*>(lds + r * BK + ((c ^ wide_kc_swz(r)) * 8));
    } else {
      const int g = lane >> 4, t = lane & 15;
      const int k = kk * 32 + 8 * g + 4 * half + (t >> 2), c = r0 + 4 * (t & 3);
      const int off = k * R + ((((c >> 3) ^ wide_mc_swz(k)) << 3) | (c & 7));
      const fp16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4f16((XFC_LDS fp16x4_t*)(lds + off));
#pragma unroll
      for (int e = 0; e < 4; ++e) f[4 * half + e] = (half_t)v[e];
    }
  }
  // The j-th read of a sub-step's fragments, in the order in which its MFMAs want them: a[0], all of b, the rest of a.
  __device__ __forceinline__ static void read_one(int j, const half_t* sa, const half_t* sb, int kk, int wm, int wn, int lane,
                                                  Frags& f) {
    constexpr int SA = A_KC ? 1 : 2;
    if (j < SA) {
      read_piece<A_KC, BM>(sa, wm * TM, kk, j, lane, f.a[0]);
    } else if (j < SA + B_RD) {
      read_piece<true, BN>(sb, wn * TN + (j - SA) * 16, kk, 0, lane, f.b[j - SA]);
    } else {
      const int q = j - B_RD;
      read_piece<A_KC, BM>(sa, wm * TM + (q / SA) * 16, kk, q % SA, lane, f.a[q / SA]);
    }
  }
  // The n-th MFMA of a sub-step, b walked back and forth so that consecutive ones share an operand register.  The
  // accumulators live in the accumulation registers ("a": with 256 of them a wave keeps 256 ordinary ones); the first
  // sub-step of a tile takes 0 as its addend instead of cleared registers (256 writes, 0.5 us a tile).  Being inline
  // asm, the instruction is invisible to the compiler's MFMA hazard bookkeeping: settle() supplies the wait states a
  // result needs before ordinary code may read it.
  template <bool FIRST>
  __device__ __forceinline__ static void mfma(int n, const Frags& f, float4v (&acc)[FM][FN]) {
    const int fm = n / FN, fn = (fm & 1) ? FN - 1 - n % FN : n % FN;
    if constexpr (FIRST)
      asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc[fm][fn]) : "v"(f.a[fm]), "v"(f.b[fn]));
    else
      asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[fm][fn]) : "v"(f.a[fm]), "v"(f.b[fn]));
  }
  // At least 18 idle issue slots must separate an MFMA from a non-MFMA read of its destination.
  __device__ __forceinline__ static void settle(float4v (&acc)[FM][FN]) {
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) asm volatile("" : "+a"(acc[fm][fn]));
  }
  // An accumulator's value for an epilogue.  Spelled out because the compiler, left to itself, copies every accumulator
  // an epilogue with branches reads to ordinary registers where the epilogue begins, and spills.
  __device__ __forceinline__ static float4v value(const float4v& acc) {
    float4v v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x;
      asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(acc[e]));
      v[e] = x;
    }
    return v;
  }
  __device__ __forceinline__ static void zero(float4v (&acc)[FM][FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  }

  // Walks the work items [item_begin, item_end) of this workgroup.
  //   get(item, oa, ob, k_begin, k_end)  fills the operands and the k range of an item (k_end > k_begin,
  //                                      k_begin a multiple of BK)
  //   epilogue(item, acc)                consumes the finished accumulators; it may use global memory and LDS
  //                                      outside the ring's LDS_BYTES, and returns whether this wave has made STORES stores at least
  // All threads of the workgroup call this together.
  //
  // Schedule per stage c: under the MFMAs of its first sub-step the fragments of the second are read and the A side
  // fetches its part of stage c+2, into the slot that stage c-1 left.  Between the sub-steps the wave waits for
  // its part of stage c+1 to have landed (all but the fetches just issued) and joins the barrier; past it, every wave has
  // finished reading stage c, so under the MFMAs of the second sub-step the B side's slot is refilled, with its part
  // of stage c+2, and the first fragments of stage c+1 are read.  What a stage does once, the ring's turns and counts, stands
  // behind a sub-step's last bump, where the matrix pipe does not wait for it.
  template <int STORES = 0, class GetItem, class Epilogue>
  __device__ __forceinline__ static void run(int item_begin, int item_end, half_t* lds, GetItem get, Epilogue epilogue) {
    if (item_begin >= item_end) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN;
    float4v acc[FM][FN];

    half_t* const a_ring = lds;
    half_t* const b_ring = lds + A_SLOTS * A_HALVES;
    Cursor<true> ca;
    Cursor<false> cb;
    ca.ring = ca.dst = lds_addr(a_ring) + (uint32_t)wave * 1024u;
    cb.ring = cb.dst = lds_addr(b_ring) + (uint32_t)wave * 1024u;
    ca.item = cb.item = item_begin;
    ca.template open<false>(get, wave, lane);
    cb.template open<false>(get, wave, lane);
    auto length = [&](int item) {  // k of an item
      Operand oa, ob;
      int kb, ke;
      get(item, oa, ob, kb, ke);
      return ke - kb;
    };
    int sa = 0, sb = 0;  // the slots of the stage being multiplied, in halves
    // Zeros in place of what that stage holds past its last k (n of them are left).  Each wave clears the pieces it
    // fetched, between its own wait for them and the barrier.
    auto clear_tail = [&](int n) {
      wait_vmcnt<0>();
      Cursor<true>::Load::clear_tail(a_ring + sa, n, wave, lane);
      Cursor<false>::Load::clear_tail(b_ring + sb, n, wave, lane);
    };
    int k_left = length(item_begin);  // k of the item from the stage being multiplied on
    // The first two stages' fetches, and the wait for the first (a loop: every line of code in front of the first MFMA costs a
    // small kernel an instruction fetch).
#pragma nounroll
    for (int stage = 0; stage < 2; ++stage) {
#pragma unroll
      for (int j = 0; j < A_CH; ++j) ca.piece(j), ca.bump(j);
#pragma unroll
      for (int j = 0; j < B_CH; ++j) cb.piece(j), cb.bump(j);
      ca.step();
      ca.template turn<false>(get, item_end, wave, lane);
      cb.step();
      cb.template turn<false>(get, item_end, wave, lane);
      if (stage == 0) {
        if (k_left < BK) clear_tail(k_left);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        wait_vmcnt_barrier<0>();
      }
    }

    Frags f0, f1;  // the fragments of a stage's first and second sub-step
#pragma unroll
    for (int j = 0; j < NR; ++j) read_one(j, a_ring + sa, b_ring + sb, 0, wm, wn, lane, f0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    int behind = 0;  // an item's first wait: 1, after the epilogue's STORES stores or more; 2, after an unknown number
    // (lambdas, not calls: written out, the compiler deals the forward kernel's scalar registers in another order)
    auto a_piece = [&](int j) { ca.piece(j); };
    auto a_bump = [&](int j) { ca.bump(j); };
    auto b_piece = [&](int j) { cb.piece(j); };
    auto b_bump = [&](int j) { cb.bump(j); };
    // The order below is the schedule: nothing may move across a sched_barrier.
    auto sub_step0 = [&](auto first_tag) {
#pragma unroll
      for (int n = 0; n < NM; ++n) {
        mfma<decltype(first_tag)::value>(n, f0, acc);
        if (n % READ_EVERY == 0 && n / READ_EVERY < NR) read_one(n / READ_EVERY, a_ring + sa, b_ring + sb, 1, wm, wn, lane, f1);
        if (n % A_EVERY == A_EVERY - 1 && n / A_EVERY < A_CH) a_piece(n / A_EVERY);
        if (n % A_EVERY == 1 && n > A_EVERY && n / A_EVERY - 1 < A_CH) a_bump(n / A_EVERY - 1);
        if (n == NM - 5) ca.step();
        if (n == NM - 4) {
          sa = sa == (A_SLOTS - 1) * A_HALVES ? 0 : sa + A_HALVES;
          pin(sa);
        }
        if (n == NM - 3) {
          sb = sb == (B_SLOTS - 1) * B_HALVES ? 0 : sb + B_HALVES;
          k_left -= BK;
          pin(sb);
          pin(k_left);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto sub_step1 = [&]() {
#pragma unroll
      for (int n = 0; n < NM; ++n) {
        mfma<false>(n, f1, acc);
        if (n % READ_EVERY == 0 && n / READ_EVERY < NR) read_one(n / READ_EVERY, a_ring + sa, b_ring + sb, 0, wm, wn, lane, f0);
        if (n % B_EVERY == B_EVERY - 1 && n / B_EVERY < B_CH) b_piece(n / B_EVERY);
        if (n % B_EVERY == 1 && n > B_EVERY && n / B_EVERY - 1 < B_CH) b_bump(n / B_EVERY - 1);
        if (n == NM - 4) cb.step();
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    for (int item = item_begin; item < item_end; ++item) {
      bool first = true, more;
      do {
        if (first) sub_step0(std::true_type{});
        else sub_step0(std::false_type{});
        first = false;
        more = k_left > 0;
        ca.template turn<true>(get, item_end, wave, lane);
        if (k_left < BK) {
          if (k_left <= 0) k_left = item + 1 < item_end ? length(item + 1) : BK;
          if (k_left < BK) clear_tail(k_left);
        }
        // this wave's LDS reads of stage c are complete (lgkmcnt) and its share of stage c+1 has landed.  After an epilogue the
        // wave's stores stand behind those fetches: where their number is known they are not waited for here (they have
        // another stage until a fetch behind them is), else, a tile's edges, the first wait drains everything.
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), in a form the compiler's own wait bookkeeping sees
        if (behind == 0) wait_lds_vmcnt_barrier<A_CH>();
        else if (behind == 1) wait_lds_vmcnt_barrier<A_CH + STORES>();
        else wait_lds_vmcnt_barrier<0>();
        behind = 0;
        sub_step1();
        cb.template turn<true>(get, item_end, wave, lane);
        // No LDS read stays pending across the loop edge (the reads above finished long before the
        // MFMAs were all issued): the compiler then knows the next stage's first MFMAs need no wait.
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      } while (more);
      settle(acc);
      if constexpr (STORES > 0) {
        behind = epilogue(item, acc) ? 1 : 2;
      } else {
        epilogue(item, acc);
        behind = 2;
      }
    }
    wait_vmcnt<0>();
  }
};

}  // namespace xfc
