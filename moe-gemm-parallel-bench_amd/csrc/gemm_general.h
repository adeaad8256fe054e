// General tile of the grouped GEMM: fp32 operands, and 16-bit operands outside the LDS-DMA layouts
// (gfx950).
//
// Operands whose inner dimension is contiguous, at any alignment and of any extent of at least 8,
// run here; the rest (other strides, negative pitches, tiny extents: general_route.h) runs GemmTile's
// element-wise staging.
//
//  * Staging.  Every thread owns fixed 8-element chunks of each K slice: 16 bytes (16-bit types) or
//    two 16-byte loads (fp32), at whatever alignment the row has (gfx950 global loads need none).
//    One to four slices are in flight in registers while another is computed from LDS.  No load is
//    predicated: a chunk that would pass the end of its row is loaded from the row's last 8
//    elements, a row past the matrix from its last row, and a slice past K from the last slice, so
//    every address stays inside the operand and the loads of a slice are the same instructions in
//    every case.  What must read as zero (k past K) is shifted or cleared when the chunk is written
//    to LDS, under uniform branches that only edge slices take.  Values past M or N feed only
//    outputs that are not stored.
//  * Layouts.  A panel whose rows run along K lives in LDS as [BX][BK], one whose rows run along M
//    or N as [BK][BX]; fragments are read as in FastTile (gemm_fast.h).  The loop is compiled for
//    each of the four combinations and chosen per problem, so transposed views cost nothing extra.
//  * fp32 on the bf16 matrix cores.  v_mfma_f32_16x16x4_f32 runs at 1/16 of the bf16 rate.  An fp32
//    value is the exact sum of three bf16 values x0 + x1 + x2 (x0 = bf16(x), x1 = bf16(x - x0),
//    x2 = x - x0 - x1: 8 + 8 + 8 significand bits), so a product needs nine bf16 products, which
//    are exact in the fp32 accumulation.  The six largest are computed; the three dropped ones
//    (x1 y2, x2 y1, x2 y2) are below 2^-25 of the product, less than the rounding of one fp32
//    addition.  TF32 operands (11 significand bits) are the exact sum of two bf16 values, and all
//    four products are computed.  Products whose parts are not both the first are summed apart from the
//    rest and added once, at the end of the tile: in one sum all parts of a product would round at the size of
//    the whole.  So sums are closer to the exact ones than the fp32 instruction's, and single products about
//    as close (error against 64 bits, fp32 instruction -> one sum of all parts -> now, normal operands, 2-norms):
//      K = 64                      1.43e-7 -> 1.07e-7 -> 4.8e-8     TF32 1.30e-7 -> 8.5e-8 -> 4.8e-8
//      K = 2048                                 7.0e-7 -> 2.7e-7              5.6e-7 -> 1.8e-7
//      rows of K = 512 with 8 values other than zero
//                                  5.4e-8 -> 1.09e-7 -> 2.9e-8      TF32 4.6e-8 -> 5.2e-8 -> 2.9e-8
//      with one                    2.54e-8 -> 3.5e-8 -> 2.60e-8     TF32 0 -> 0 -> 0
//    and the same at scales down to products of 2^-125, whose subnormal parts the matrix cores keep.  It
//    costs up to 7 % on large calls (8 x [512,2048]@[2048,1536] 152 -> 154 us, 4 x [2048,4096]@[4096,4096]
//    1382 -> 1403 us, TF32 1071 -> 1097 us).  Below K = 8 the fp32 instruction runs.
//    Chunks are split on their way into LDS, once per workgroup, into one LDS panel per part.
//  * Bound and measured.  Large fp32 tiles are bound by the matrix cores and by the split's vector
//    instructions (about 7.5 an element in IEEE mode, 7 in TF32), so the eight-wave 256x128 tile, which
//    splits each element for twice the MFMAs of a 64-wide tile, leads: 4 x [2048,4096]@[4096,4096] runs at
//    196 to 202 TFLOP/s by card (1176 to 1211 of bf16 MFMA work; matrix cores busy in 57 % of the cycles, vector
//    issue in 35 %), TF32 at 250 (46 and 49 % on 128x128 tiles); the fp32 instruction's nominal peak is 157.
//    8 x [512,2048]@[2048,1536] 459 -> 160 us (192 tiles on 256 CUs: 39 and 25 %); TF32 [1024,4096]@[4096,3584]
//    676 -> 132 us.  16-bit tiles are bound by the latency of a slice's loads where few workgroups share a
//    CU: fp16 [777,2881]@[2881,1443] 148 -> 39 us whole, 28 in three splits (element-wise gathers before),
//    with the matrix cores busy in 8 %; bf16 [4001,4003]@[4003,4005] runs at 854 to 873 TFLOP/s.
//  * Split-K.  Few tiles leave the chip idle, and a lone workgroup on a CU runs at the latency of its
//    steps, so a tile's K slices can be shared by several workgroups (fp32 [64,4096]@[4096,1024]:
//    64 us whole, 17 us in sixteen; the reduction costs about 5 us, so large groups stay whole): each
//    stores its fp32 partial, and the last to arrive sums them in split order (deterministic) and stores C.
//    Counters, partial layout and coherence are FastTile's (gemm_fast.h, split_store); nobody waits for
//    another unit.
//  * Range.  The split is exact and its products neither overflow nor lose their small parts while
//    every non-zero operand lies in [2^-96, 2^60).  Each thread keeps the extremes of what it
//    loaded, and the accumulators show overflow.  A tile with smaller values reads its operands' largest
//    value and keeps its sums if what the small ones may lack cannot show in any output (small_shows): a few
//    such values among ordinary ones cost 12 to 29 % (fp32 [4096,2048]@[2048,1536] 153 -> 184 us,
//    [1024,2048]@[2048,1536] 55 -> 70; the fp32 instruction alone 307 and 95).  A tile whose outputs are as
//    small or zero, and one with infinities, NaN or (TF32) values from 2^60, is computed again by GemmTile
//    with the fp32 instruction, a split unit over its own part of K; that is up to 2.3 times slower than a
//    kernel of it alone ([1024,2048]@[2048,1536] with an infinity in every tile: 185 us against 95).
#pragma once

#include "gemm_fast.h"
#include "gemm_kernel.h"
#include "general_route.h"

namespace moegemm {

typedef uint32_t u32x4_a2_t __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4_a4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a2_t __attribute__((ext_vector_type(2), aligned(2)));

// PARTS: bf16 panels per operand (3 = fp32 operands, 2 = TF32 operands, 1 = 16-bit operands).
template <class E, int BM_, int BN_, int BK_, int WM_, int WN_, int PARTS_>
struct GeneralTile {
  using Plain = GemmTile<E, BM_, BN_, BK_, WM_, WN_, true>;
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, PARTS = PARTS_;
  static constexpr bool F32 = E::is_f32;
  static constexpr int ES = sizeof(typename E::raw);
  static constexpr int NW = WM * WN;
  static constexpr int NT = NW * 64;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int MI = (WTM >= 32 && WTN >= 32) ? 32 : 16;
  static constexpr int MIK = MI == 32 ? 16 : 32;
  static constexpr int KK = BK / MIK;
  static constexpr int FM = WTM / MI, FN = WTN / MI;
  static constexpr int ACC = MI * MI / 64;
  static constexpr int PRODUCTS = PARTS == 3 ? 6 : PARTS * PARTS;  // MFMAs per fragment pair and K step
  static constexpr int LM = PARTS > 1 ? FM : 1, LN = PARTS > 1 ? FN : 1;  // sums of the small products
  // Two sums of 64 registers and all of a K step's fragments are more than a wave's registers hold.
  static constexpr bool TIGHT = PARTS == 3 && FM * FN * ACC >= 64 && NW == 8;
  static constexpr int VL = ES / 2;  // 16-byte loads per 8-element chunk
  static constexpr int A_CHUNKS = BM * BK / 8, B_CHUNKS = BK * BN / 8;
  static constexpr int A_PT = (A_CHUNKS + NT - 1) / NT, B_PT = (B_CHUNKS + NT - 1) / NT;
  // Slices in flight in registers: one where a slice's MFMAs outlast a load, else two or, where a
  // slice is small, four.
  static constexpr int SLICE_REGS = (A_PT + B_PT) * VL * 4;
  static constexpr int DEPTH = KK * FM * FN * PRODUCTS * (MI == 32 ? 2 : 1) >= 48 ? 1 : SLICE_REGS <= 16 ? 4 : 2;
  static constexpr int UNROLL = DEPTH > 2 ? DEPTH : 2;  // steps per loop: LDS buffer and register set are static
  static constexpr int A_BYTES = A_CHUNKS * 16, B_BYTES = B_CHUNKS * 16;  // one part
  static constexpr int STAGE_BYTES = PARTS * (A_BYTES + B_BYTES);
  static constexpr int PREFIX = Plain::PREFIX;
  static constexpr int PREFIX_OFFSET = 2 * STAGE_BYTES > Plain::PREFIX_OFFSET ? 2 * STAGE_BYTES : Plain::PREFIX_OFFSET;
  static constexpr int LDS_BYTES = PREFIX_OFFSET + (PREFIX + 1) * 4 + NT * 4;
  // Tiles of four waves whose LDS fits twice run two workgroups a CU: 256 registers a wave.
  static constexpr int WAVES_PER_EU = 2 * LDS_BYTES <= 160 * 1024 || NW == 8 ? 2 : 1;
  static constexpr bool CHAIN_OK = false;
  static constexpr bool CHAIN_STEALING = false;
  static constexpr bool ABSOLUTE_K = true;

  static_assert(F32 ? PARTS >= 2 : PARTS == 1, "16-bit operands are one part, fp32 operands two or three");
  static_assert(BK % MIK == 0 && WTM % MI == 0 && WTN % MI == 0, "tile shape");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget of one CU");

  using acc_t = typename std::conditional<ACC == 16, f32x16_t, f32x4_t>::type;
  using vec_t = typename std::conditional<F32, u32x4_a4_t, u32x4_a2_t>::type;

  // One operand's chunks of this thread.  XC: rows run along the operand's M or N dimension x.
  // Global addresses are a uniform base plus an unsigned 32-bit offset (chunk_route checked the pitch).
  template <bool XC, int BX, int PT>
  struct Operand {
    static constexpr int CPR = XC ? BX / 8 : BK / 8;  // chunks per LDS row
    static constexpr int CHUNKS = BX * BK / 8;
    // Chunk i lies i * NT / CPR rows below chunk 0 in the same LDS column; where that keeps the row's
    // swizzle, the chunks share one LDS address.
    static constexpr int RSTEP = NT / CPR;
    static constexpr bool SHARED = NT % CPR == 0 && RSTEP % (XC ? 16 : 32) == 0 && CHUNKS % NT == 0;
    const char* base;    // row x0 (K-contiguous) or column x0 (XC) of the matrix; uniform
    uint32_t off[PT];    // K-contiguous: offset of the chunk's row, inside the matrix; XC: of its column
    int32_t col;         // first chunk's position along the LDS row, in elements
    uint32_t pitch;      // bytes between K rows (XC)
    uint32_t lds[SHARED ? 1 : PT];
    int32_t k, x_over;   // x_over: elements of the tile's partial x chunk past the matrix (XC), 0 if none
    int32_t x_limit;     // matrix extent along x, relative to the tile

    __device__ static __forceinline__ void place(int i, int& r, int& c) {
      int cl = (int)threadIdx.x + i * NT;
      if (CHUNKS % NT != 0) cl = min(cl, CHUNKS - 1);
      r = cl / CPR;
      c = cl % CPR;
    }

    __device__ __forceinline__ void setup(const char* p, int64_t sx, int64_t sk, int x0, int extent, int32_t k_) {
      k = k_;
      x_limit = extent - x0;
      x_over = XC && x_limit < BX ? (8 - (x_limit & 7)) & 7 : 0;
      pitch = XC ? (uint32_t)(sk * ES) : 0;
      // The last 8 columns may start before x0: the base steps back with them.
      const int back = XC ? max(0, 8 - x_limit) : 0;
      base = p + (XC ? (int64_t)(x0 - back) * ES : (int64_t)x0 * sx * ES);
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        int r, c;
        place(i, r, c);
        if (i == 0) col = c * 8;
        off[i] = XC ? (uint32_t)(min(c * 8, x_limit - 8) + back) * ES
                    : (uint32_t)min(r, x_limit - 1) * (uint32_t)(sx * ES);
        if (!SHARED || i == 0) lds[i] = (uint32_t)(r * CPR + (c ^ (XC ? swz_b(r, CPR) : swz_a(r, CPR)))) * 16u;
      }
    }

    // Loads of the slice that starts at k0 < k.
    __device__ __forceinline__ void load(u32x4_t (&out)[PT][VL], int k0) const {
      const char* from = XC ? base + (int64_t)k0 * pitch : base;
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        int r, c;
        place(i, r, c);
        const uint32_t at = XC ? off[i] + (uint32_t)min(r, k - 1 - k0) * pitch
                               : off[i] + (uint32_t)min(k0 + (SHARED ? col : c * 8), k - 8) * (uint32_t)ES;
#pragma unroll
        for (int v = 0; v < VL; ++v) out[i][v] = *MOEGEMM_GLOBAL(const vec_t, from + (uint64_t)at + v * 16);
      }
    }

    // Writes the chunks to the slice's LDS panel (PARTS of them).  EDGE false: the slice lies inside K
    // and the tile has no partial x chunk.
    template <bool EDGE>
    __device__ __forceinline__ void store(u32x4_t (&in)[PT][VL], int k0, char* panel, uint32_t (&range)[2]) const {
      const bool edge = EDGE && (k0 + BK > k || x_over != 0);  // uniform
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        if (edge) {
          int r, c;
          place(i, r, c);
          const int over = XC ? x_over : (8 - (k & 7)) & 7;
          const int past = XC ? c * 8 + 8 - x_limit : k0 + c * 8 + 8 - k;
          if (past > 0 && past < 8) shift_down(in[i], over);
          const bool clear = XC ? k0 + r >= k : past >= 8;
          if (clear) {
#pragma unroll
            for (int v = 0; v < VL; ++v) in[i][v] = u32x4_t{0u, 0u, 0u, 0u};
          }
        }
        u32x4_t part[PARTS];
        split(in[i], part, range);
        char* dst = panel + (SHARED ? lds[0] : lds[SHARED ? 0 : i]) + (SHARED ? i * RSTEP * CPR * 16 : 0);
        if (CHUNKS % NT == 0 || (int)threadIdx.x + i * NT < CHUNKS) {
#pragma unroll
          for (int q = 0; q < PARTS; ++q) *reinterpret_cast<u32x4_t*>(dst + q * (BX * BK * 2)) = part[q];
        }
      }
    }
  };

  // Moves a chunk's elements down by `over` (uniform, 1 to 7), zeros in at the top.
  __device__ static __forceinline__ void shift_down(u32x4_t (&v)[VL], int over) {
    uint32_t w[4 * VL];
#pragma unroll
    for (int i = 0; i < 4 * VL; ++i) w[i] = v[i / 4][i % 4];
    const int words = F32 ? over : over >> 1;
#pragma unroll
    for (int bit = 4 * VL / 2; bit >= 1; bit >>= 1)
      if (words & bit) {
#pragma unroll
        for (int i = 0; i < 4 * VL; ++i) w[i] = i + bit < 4 * VL ? w[(i + bit) % (4 * VL)] : 0u;
      }
    if (!F32 && (over & 1)) {
#pragma unroll
      for (int i = 0; i < 4 * VL; ++i) w[i] = (w[i] >> 16) | (i + 1 < 4 * VL ? w[(i + 1) % (4 * VL)] << 16 : 0u);
    }
#pragma unroll
    for (int i = 0; i < 4 * VL; ++i) v[i / 4][i % 4] = w[i];
  }

  __device__ static __forceinline__ uint32_t pack_bf16(float x, float y) {
    uint32_t h;  // one instruction; the compiler converts the halves one by one and merges them
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(h) : "v"(x), "v"(y));
    return h;
  }

  // The chunk's bf16 parts.  range[1]: the smallest non-zero |x| seen (as twice its bits, less one: zero
  // wraps to the top).  range[0], TF32 only: the largest |x| (as float bits; a NaN stays), because
  // rounding can turn a NaN into a number.  In IEEE mode large values need no watch: whatever
  // overflows in the parts or their products (infinities and NaN too) leaves an accumulator that is
  // not finite (all_finite).  The register it saves ended most spills of the 256x128 loop (185 -> 157 us on
  // 8 x [512,2048]@[2048,1536] when it went).
  __device__ static __forceinline__ void split(const u32x4_t (&in)[VL], u32x4_t (&part)[PARTS], uint32_t (&range)[2]) {
    if constexpr (!F32) {
      part[0] = in[0];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t u0 = in[(2 * i) / 4][(2 * i) % 4], u1 = in[(2 * i + 1) / 4][(2 * i + 1) % 4];
        if constexpr (PARTS == 2) asm("v_maximum3_f32 %0, %0, |%1|, |%2|" : "+v"(range[0]) : "v"(u0), "v"(u1));
        range[1] = min(min(range[1], (u0 << 1) - 1u), (u1 << 1) - 1u);
        if constexpr (PARTS == 2) {  // TF32: 10-bit mantissa, ties away (NaN leaves by its range)
          u0 = (u0 + 0x1000u) & 0xffffe000u;
          u1 = (u1 + 0x1000u) & 0xffffe000u;
        }
        float x = __builtin_bit_cast(float, u0), y = __builtin_bit_cast(float, u1);
#pragma unroll
        for (int q = 0; q < PARTS; ++q) {
          const uint32_t h = pack_bf16(x, y);
          part[q][i] = h;
          x -= __builtin_bit_cast(float, h << 16);
          y -= __builtin_bit_cast(float, h & 0xffff0000u);
        }
      }
    }
  }
  __device__ static __forceinline__ bool all_finite(const acc_t (&acc)[FM][FN]) {
    float worst = 0.0f;  // x - x is zero exactly when x is finite
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int i = 0; i < ACC; ++i) worst += acc[fm][fn][i] - acc[fm][fn][i];
    return worst == 0.0f;
  }
  __device__ static __forceinline__ float block_max(uint32_t bits) {
    __shared__ uint32_t s_max;
    if (threadIdx.x == 0) s_max = 0;
    __syncthreads();
    atomicMax(&s_max, bits);
    __syncthreads();
    return __builtin_bit_cast(float, s_max);
  }
  // Whether what the parts lose of values below 2^-96 may show in an output of this lane.  Such a value is
  // held to within 2^-125 (its parts below the smallest normal number may be lost), and a product of parts to
  // within 2^-126, so a sum of `depth` products of values up to `peak` is off by less than
  // depth * 2^-123 * (1 + 2 peak).  That is an eighth of a unit in the last place of any output from 2^27 times as
  // much on; smaller outputs, zeros among them, ask for the fp32 instruction.
  __device__ static __forceinline__ bool small_shows(const acc_t (&acc)[FM][FN], const ProblemDesc& pd, int m0, int n0,
                                                     int wave_m, int wave_n, int depth, float peak) {
    const int lane = threadIdx.x & 63;
    const int row0 = m0 + wave_m * WTM + lane % MI;
    const int col0 = n0 + wave_n * WTN + ((MI == 32) ? (lane >> 5) * 4 : (lane >> 4) * 4);
    float least = __builtin_inff();
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int i = 0; i < ACC; ++i) {
          const int gn = col0 + fn * MI + (i / 4) * 8 + i % 4;
          const bool stored = row0 + fm * MI < pd.m && gn < pd.n;
          least = __builtin_fminf(least, stored ? __builtin_fabsf(acc[fm][fn][i]) : __builtin_inff());
        }
    return least < (float)depth * 0x1p-96f * (1.0f + 2.0f * peak);
  }
  // Bits of 2^60, and twice those of 2^-96 less one.
  static constexpr uint32_t kTooLarge = (127u + 60u) << 23;
  static constexpr uint32_t kTooSmall = ((127u - 96u) << 24) - 1u;

  // Fragments of one operand (as FastTile's frag_rows / frag_transposed): per-lane LDS offsets of the
  // wave's first rows, to which fragment and K step add constants (the swizzles do not see them).
  template <bool XC, int BX, int NF>
  struct Frags {
    static constexpr int CPR = XC ? BX / 8 : BK / 8;
    // Fragments 16 rows apart differ in a swizzle bit when a K-contiguous row has 8 chunks.
    static constexpr int ROWS = !XC && MI == 16 && CPR == 8 ? NF : 1;
    uint32_t off[XC ? NF : KK * ROWS];

    __device__ __forceinline__ void setup(int x0) {
      const int lane = threadIdx.x & 63;
      if constexpr (!XC) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
          for (int f = 0; f < ROWS; ++f) {
            const int row = x0 + f * MI + (lane % MI);
            off[kk * ROWS + f] = (uint32_t)(row * CPR + (((kk * MIK) / 8 + lane / MI) ^ swz_a(row, CPR))) * 16u;
          }
      } else {
        const int g = lane >> 4, s = lane & 15;
        const int row = MI == 32 ? 8 * (g >> 1) + (s >> 2) : 8 * g + (s >> 2);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const int col = x0 + f * MI + (MI == 32 ? 16 * (g & 1) + 4 * (s & 3) : 4 * (s & 3));
          off[f] = (uint32_t)((row * CPR + ((col >> 3) ^ swz_b(row, CPR))) * 16 + (col & 7) * 2);
        }
      }
    }
    __device__ __forceinline__ i16x8_t get(const char* panel, int f, int kk) const {
      if constexpr (!XC) {
        const char* p = panel + off[kk * ROWS + (ROWS > 1 ? f : 0)] + (ROWS > 1 ? 0 : f * MI * CPR * 16);
        return *reinterpret_cast<const i16x8_t*>(p);
      } else {
        const char* p0 = panel + off[f] + kk * MIK * CPR * 16;
        const char* p1 = p0 + 4 * CPR * 16;
        i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(p0));
        i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(p1));
        return i16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
  };

  __device__ static __forceinline__ acc_t mfma(i16x8_t b, i16x8_t a, acc_t c) {
    if constexpr (E::dtype == DT_F16) {
      if constexpr (MI == 32)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, b), __builtin_bit_cast(f16x8_t, a), c, 0, 0, 0);
      else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, b), __builtin_bit_cast(f16x8_t, a), c, 0, 0, 0);
    } else {
      if constexpr (MI == 32)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), c, 0, 0, 0);
      else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), c, 0, 0, 0);
    }
  }

  // Fragment registers of one K step; four-wave tiles read all of a slice's fragments ahead of its MFMAs
  // where they fit (a lone wave on its SIMD has nothing else to hide the LDS latency of each K step).
  static constexpr int STEP_REGS = PARTS * (FM + FN) * 4;
  static constexpr bool READ_AHEAD =
      NW <= 4 && KK * STEP_REGS + FM * FN * ACC + DEPTH * SLICE_REGS <= (WAVES_PER_EU == 1 ? 320 : 160);

  // Products whose parts are not both the first go to sums of their own: those parts then round into a sum
  // of their size, and the first parts' products, which have 16 significant bits, hardly round at all.
  template <class FA, class FB>
  __device__ static __forceinline__ void compute(acc_t (&acc)[FM][FN], acc_t (&low)[LM][LN], const char* lds,
                                                 const FA& fa, const FB& fb) {
    i16x8_t af[KK][PARTS][FM], bf[KK][PARTS][FN];
    auto read_a = [&](int kk, int q) {
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) af[kk][q][fm] = fa.get(lds + q * A_BYTES, fm, kk);
    };
    auto read_b = [&](int kk, int q) {
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) bf[kk][q][fn] = fb.get(lds + PARTS * A_BYTES + q * B_BYTES, fn, kk);
    };
    auto multiply = [&](int kk, int qa, int qb) {
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
          acc_t& to = qa + qb > 0 ? low[fm % LM][fn % LN] : acc[fm][fn];
          to = mfma(bf[kk][qb][fn], af[kk][qa][fm], to);
        }
    };
    constexpr int kMemoryMayCross = 0x0216;  // vector, scalar, global memory and LDS writes may cross
    if constexpr (READ_AHEAD) {
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
#pragma unroll
        for (int q = 0; q < PARTS; ++q) {
          read_a(kk, q);
          read_b(kk, q);
        }
      __builtin_amdgcn_sched_barrier(kMemoryMayCross);
    }
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      if constexpr (TIGHT) {  // A's parts one ahead of their products
        read_a(kk, 2);
        read_b(kk, 0);
        read_a(kk, 1);
        read_b(kk, 1);
        read_b(kk, 2);
        __builtin_amdgcn_sched_barrier(kMemoryMayCross);
        multiply(kk, 2, 0);
        read_a(kk, 0);
        __builtin_amdgcn_sched_barrier(kMemoryMayCross);
        multiply(kk, 1, 1);
        multiply(kk, 1, 0);
        multiply(kk, 0, 2);
        multiply(kk, 0, 1);
        multiply(kk, 0, 0);
      } else {
        if constexpr (!READ_AHEAD) {
#pragma unroll
          for (int q = 0; q < PARTS; ++q) {
            read_a(kk, q);
            read_b(kk, q);
          }
        }
        // Products in falling order of the parts' sum: the small ones are added first.
#pragma unroll
        for (int sum = PARTS == 3 ? 2 : 2 * (PARTS - 1); sum >= 0; --sum)
#pragma unroll
          for (int qa = 0; qa < PARTS; ++qa) {
            const int qb = sum - qa;
            if (qb >= 0 && qb < PARTS) multiply(kk, qa, qb);
          }
      }
    }
  }

  // C: four consecutive columns a lane (see GemmTile::store_tile), stored at any alignment.
  __device__ static __forceinline__ void store_tile(const acc_t (&acc)[FM][FN], const ProblemDesc& pd, int m0, int n0,
                                                    int wave_m, int wave_n) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      const int gm = m0 + wave_m * WTM + fm * MI + (lane % MI);
      if (gm >= pd.m) continue;
      char* crow = pd.c + (int64_t)gm * pd.scm * ES;
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int q = 0; q < ACC / 4; ++q) {
          const int gn = n0 + wave_n * WTN + fn * MI + ((MI == 32) ? (q * 8 + (lane >> 5) * 4) : ((lane >> 4) * 4));
          const f32x4_t v = {acc[fm][fn][q * 4 + 0], acc[fm][fn][q * 4 + 1], acc[fm][fn][q * 4 + 2],
                             acc[fm][fn][q * 4 + 3]};
          if (pd.scn == 1 && gn + 4 <= pd.n) {
            if constexpr (F32)
              *MOEGEMM_GLOBAL(u32x4_a4_t, crow + (int64_t)gn * 4) = __builtin_bit_cast(u32x4_t, v);
            else
              *MOEGEMM_GLOBAL(u32x2_a2_t, crow + (int64_t)gn * 2) = pack4<E>(v);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (gn + e < pd.n) store1<E>(crow + (int64_t)(gn + e) * pd.scn * ES, v[e]);
          }
        }
    }
  }

  // Split-K.  A unit's fp32 partial: 16-byte accumulator chunks in the order of acc, 64 lanes each.
  static constexpr int CHUNKS = FM * FN * (ACC / 4);  // chunks per lane
  __device__ static __forceinline__ auto partial(const ProblemDesc& pd, int split) {
    return __builtin_amdgcn_make_buffer_rsrc(pd.partials + ((int64_t)pd.slot0 + split) * (BM * BN), (short)0,
                                             BM * BN * 4, (int)kBufferFlags);
  }
  __device__ static __forceinline__ void store_partial(const acc_t (&acc)[FM][FN], const ProblemDesc& pd) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane_off = (wave * CHUNKS * 64 + (int)(threadIdx.x & 63)) * 16;
    const auto mine = partial(pd, pd.split);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const acc_t& t = acc[c / (ACC / 4) / FN][c / (ACC / 4) % FN];
      const int q = c % (ACC / 4);
      const f32x4_t v = {t[q * 4 + 0], t[q * 4 + 1], t[q * 4 + 2], t[q * 4 + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(v, mine, lane_off + c * 1024, 0, kDeviceCoherent);
    }
  }
  // The same of a unit that left the split's range, by the fp32 instruction.  Both layouts give a lane four
  // consecutive columns at a time, so whole chunks change places.
  __device__ static __forceinline__ void store_plain_partial(const ProblemDesc& pd, int tm, int tn, char* smem,
                                                             bool tf32) {
    ProblemDesc unit = pd;
    unit.a += (int64_t)pd.k_begin * pd.sak * ES;
    unit.b += (int64_t)pd.k_begin * pd.sbk * ES;
    unit.k = pd.k_end - pd.k_begin;
    typename Plain::acc_t sums[Plain::FM][Plain::FN];
    Plain::accumulate(sums, unit, tm, tn, smem, tf32);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const auto mine = partial(pd, pd.split);
#pragma unroll
    for (int fm = 0; fm < Plain::FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < Plain::FN; ++fn) {
        const int row = fm * 16 + lane % 16, col = fn * 16 + lane / 16 * 4;  // in the wave's sub-tile
        const int chunk = (row / MI * FN + col / MI) * (ACC / 4) + (MI == 32 ? col % 32 / 8 : 0);
        const int holder = MI == 32 ? row % 32 + col % 8 / 4 * 32 : lane;
        const auto& t = sums[fm][fn];
        const f32x4_t v = {t[0], t[1], t[2], t[3]};
        const int at = ((wave * CHUNKS + chunk) * 64 + holder) * 16;
        __builtin_amdgcn_raw_buffer_store_b128(v, mine, at, 0, kDeviceCoherent);
      }
  }
  // Arrives at the tile's counter.  The last unit to do so re-arms it, sums the partials into acc in split
  // order, and returns true.
  __device__ static __forceinline__ bool reduce_splits(acc_t (&acc)[FM][FN], const ProblemDesc& pd) {
    __shared__ int s_last;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane_off = (wave * CHUNKS * 64 + (int)(threadIdx.x & 63)) * 16;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      int32_t* word = pd.counters + pd.tile;
      s_last = atomicAdd(word, 1) == pd.splits - 1;
      if (s_last) atomicExch(word, 0);
    }
    __syncthreads();
    if (!uniform(s_last)) return false;
    constexpr int GC = CHUNKS < 4 ? CHUNKS : 4, WAYS = 4;  // chunks and partials read at a time
#pragma unroll
    for (int c0 = 0; c0 < CHUNKS; c0 += GC) {
      f32x4_t sum[GC];
#pragma unroll
      for (int i = 0; i < GC; ++i) sum[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      for (int s0 = 0; s0 < pd.splits; s0 += WAYS) {
        f32x4_t v[WAYS][GC];
#pragma unroll
        for (int w = 0; w < WAYS; ++w) {
          const auto from = partial(pd, min(s0 + w, pd.splits - 1));
#pragma unroll
          for (int i = 0; i < GC; ++i)
            v[w][i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                      from, lane_off + (c0 + i) * 1024, 0, kDeviceCoherent));
        }
#pragma unroll
        for (int w = 0; w < WAYS; ++w)
          if (s0 + w < pd.splits) {
#pragma unroll
            for (int i = 0; i < GC; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) sum[i][e] += v[w][i][e];
          }
      }
#pragma unroll
      for (int i = 0; i < GC; ++i) {
        const int c = c0 + i;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[c / (ACC / 4) / FN][c / (ACC / 4) % FN][c % (ACC / 4) * 4 + e] = sum[i][e];
      }
    }
    return true;
  }

  // The sums of the tile (split-K: of the unit's K range) with both operands in 8-element chunks; false when
  // Plain must compute them.
  template <bool AT, bool BT, int EPI>
  __device__ static __forceinline__ bool chunk_tile(acc_t (&acc)[FM][FN], const ProblemDesc& pd, int tm, int tn,
                                                    char* smem) {
    const int wave = threadIdx.x >> 6;
    const int wave_m = wave / WN, wave_n = wave % WN;
    const int m0 = tm * BM, n0 = tn * BN;
    Operand<AT, BM, A_PT> a;
    Operand<!BT, BN, B_PT> b;
    a.setup(pd.a, pd.sam, pd.sak, m0, pd.m, pd.k);
    b.setup(pd.b, pd.sbn, pd.sbk, n0, pd.n, pd.k);
    Frags<AT, BM, FM> fa;
    Frags<!BT, BN, FN> fb;
    fa.setup(wave_m * WTM);
    fb.setup(wave_n * WTN);
    acc_t low[LM][LN];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int i = 0; i < ACC; ++i) acc[fm][fn][i] = low[fm % LM][fn % LN][i] = 0.0f;
    uint32_t range[2] = {0u, 0xffffffffu};

    // K slices first .. first + last, from k_first on; a unit's range starts at a whole slice.
    const int k_first = EPI == EPI_SPLIT ? pd.k_begin : 0, k_end = EPI == EPI_SPLIT ? pd.k_end : pd.k;
    const int last = (k_end - k_first + BK - 1) / BK - 1;
    u32x4_t ra[DEPTH][A_PT][VL], rb[DEPTH][B_PT][VL];
    // Register set of slice kt: kt % DEPTH; LDS buffer: kt % 2.  J: kt modulo UNROLL.
    auto load = [&](auto j, int kt) {
      constexpr int S = decltype(j)::value % DEPTH;
      const int k0 = k_first + min(kt, last) * BK;
      a.load(ra[S], k0);
      b.load(rb[S], k0);
    };
    auto store = [&](auto j, auto edge, int kt) {
      constexpr int S = decltype(j)::value % DEPTH;
      constexpr bool EDGE = decltype(edge)::value;
      char* lds = smem + (decltype(j)::value % 2) * STAGE_BYTES;
      a.template store<EDGE>(ra[S], k_first + kt * BK, lds, range);
      b.template store<EDGE>(rb[S], k_first + kt * BK, lds + PARTS * A_BYTES, range);
    };
    // Slice kt is computed from its LDS buffer while slice kt + 1 (in registers) goes to the other
    // one and slices up to kt + DEPTH are in flight.  Steps whose stored slice is no edge are one
    // basic block, so the split's vector instructions can issue between the MFMAs.
    auto step = [&](auto j, auto edge, int kt) {
      constexpr int J = decltype(j)::value;
      using ahead = std::integral_constant<int, (J + DEPTH) % UNROLL>;
      using next = std::integral_constant<int, (J + 1) % UNROLL>;
      load(ahead{}, kt + DEPTH);
      compute(acc, low, smem + (J % 2) * STAGE_BYTES, fa, fb);
      store(next{}, edge, kt + 1);
      __syncthreads();
    };
    // Steps kt .. kt + UNROLL - 1, those before `end`.
    auto steps = [&](auto edge, int kt, int end) {
      step(std::integral_constant<int, 0>{}, edge, kt);
      if (!decltype(edge)::value || kt + 1 < end) step(std::integral_constant<int, 1>{}, edge, kt + 1);
      if constexpr (UNROLL == 4) {
        if (!decltype(edge)::value || kt + 2 < end) step(std::integral_constant<int, 2>{}, edge, kt + 2);
        if (!decltype(edge)::value || kt + 3 < end) step(std::integral_constant<int, 3>{}, edge, kt + 3);
      }
    };
    load(std::integral_constant<int, 0>{}, 0);
    if constexpr (DEPTH >= 2) load(std::integral_constant<int, 1>{}, 1);
    if constexpr (DEPTH == 4) {
      load(std::integral_constant<int, 2>{}, 2);
      load(std::integral_constant<int, 3>{}, 3);
    }
    store(std::integral_constant<int, 0>{}, std::true_type{}, 0);
    __syncthreads();
    int kt = 0;
    if (a.x_over == 0 && b.x_over == 0) {
      const int inner = (k_end - k_first) / BK;  // whole slices
      for (; kt + UNROLL < inner; kt += UNROLL) steps(std::false_type{}, kt, 0);
    }
    for (; kt < last; kt += UNROLL) steps(std::true_type{}, kt, last);
    compute(acc, low, smem + (last & 1) * STAGE_BYTES, fa, fb);
    bool bad = false;
    if constexpr (F32) {
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int i = 0; i < ACC; ++i) acc[fm][fn][i] += low[fm % LM][fn % LN][i];
      const bool past = PARTS == 2 ? range[0] >= kTooLarge : !all_finite(acc);
      // Also the barrier between this tile's LDS reads and the next tile's writes.
      if (__syncthreads_or(past || range[1] < kTooSmall)) {
        bad = __syncthreads_or(past) != 0;
        if (!bad) {  // small values only: do they show in an output?
          uint32_t peak = 0;  // largest |x|, as float bits
#pragma unroll 4
          for (int kt = 0; kt <= last; ++kt) {
            u32x4_t va[A_PT][VL], vb[B_PT][VL];
            a.load(va, k_first + kt * BK);
            b.load(vb, k_first + kt * BK);
#pragma unroll
            for (int v = 0; v < VL * 4; ++v) {
#pragma unroll
              for (int i = 0; i < A_PT; ++i) peak = max(peak, va[i][v / 4][v % 4] & 0x7fffffffu);
#pragma unroll
              for (int i = 0; i < B_PT; ++i) peak = max(peak, vb[i][v / 4][v % 4] & 0x7fffffffu);
            }
          }
          bad = __syncthreads_or(small_shows(acc, pd, m0, n0, wave_m, wave_n, k_end - k_first, block_max(peak))) != 0;
        }
      }
    } else {
      __syncthreads();
    }
    return !bad;
  }

  template <int EPI, class Hook>
  __device__ static __forceinline__ void run_tile(const ProblemDesc& pd, int tm, int tn, char* smem, bool tf32,
                                                  Hook&& before_store) {
    static_assert(EPI == EPI_C || EPI == EPI_SPLIT, "the general kernel has no stream-K tail");
    if (pd.swiglu || (EPI == EPI_C && pd.splits > 1)) return;  // the host launches neither
    const ChunkRoute r = chunk_route(F32, ES, BM, BN, pd.m, pd.n, pd.k, pd.sam, pd.sak, pd.sbk, pd.sbn);
    acc_t acc[FM][FN];
    // Whole tiles share one copy of what follows their K loops, after all four loops; split units store their
    // partials within each and share the reduction.  Otherwise that code took registers from the loops: fp32
    // 256x128 spilled 382 of them and keeps 89 this way, 16-bit split 256x256 1228 and 103.
    auto run = [&](auto at, auto bt) {
      if constexpr (EPI == EPI_SPLIT) {
        acc_t sums[FM][FN];
        const bool ok = chunk_tile<decltype(at)::value, decltype(bt)::value, EPI>(sums, pd, tm, tn, smem);
        if (ok) store_partial(sums, pd);
        return ok;
      } else {
        return chunk_tile<decltype(at)::value, decltype(bt)::value, EPI>(acc, pd, tm, tn, smem);
      }
    };
    using yes = std::true_type;
    using no = std::false_type;
    bool done = false;
    if (r.a_rows && r.b_cols) {
      done = run(no{}, no{});
    } else if (r.a_rows && r.b_rows) {
      done = run(no{}, yes{});
    } else if (r.a_cols && (r.b_cols || r.b_rows)) {
      if constexpr (BM >= 32) done = r.b_cols ? run(yes{}, no{}) : run(yes{}, yes{});
    }
    if constexpr (EPI == EPI_SPLIT) {
      if ((r.a_rows || (BM >= 32 && r.a_cols)) && (r.b_rows || r.b_cols)) {
        if constexpr (F32) {
          if (!done) store_plain_partial(pd, tm, tn, smem, tf32);
        }
        if (!reduce_splits(acc, pd)) return;
        done = true;
      } else if (pd.split != 0) {
        return;  // operands Plain must stage: unit 0 of each tile computes it whole
      }
    }
    if (done) {
      before_store();
      const int wave = threadIdx.x >> 6;
      store_tile(acc, pd, tm * BM, tn * BN, wave / WN, wave % WN);
    } else {
      ProblemDesc whole = pd;
      whole.splits = 1;
      Plain::template run_tile<EPI_C>(whole, tm, tn, smem, tf32, before_store);
    }
  }
};

}  // namespace moegemm
