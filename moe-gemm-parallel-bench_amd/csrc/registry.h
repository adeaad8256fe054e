// Table of compiled kernel instantiations.  Each entry is one tile configuration for one dtype,
// with up to two kernels: the LDS-DMA fast path (16-bit operands in vector layouts) and the
// general register-staged kernel (any strides/alignment, and all fp32 work).
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_fast.h"
#include "gemm_general.h"
#include "gemm_kernel.h"
#include "gemm_pingpong.h"

namespace moegemm {

typedef hipError_t (*LaunchFn)(const KParams&, int grid, hipStream_t stream);

struct KernelEntry {
  int dtype;
  int block_m, block_n, block_k;
  int num_warps;   // wave64 wavefronts per workgroup
  int num_stages;  // LDS stages of the fast path's K pipeline
  int waves_m, waves_n;
  int lds_bytes;   // fast path if present, else general
  int swiglu_ok;   // the fast path can run the packed Gate+Up SwiGLU epilogue (even FN)
  LaunchFn launch_fast;     // null when the dtype has no fast path
  LaunchFn launch_general;
  LaunchFn launch_fast_split;  // the fast path's split-K kernel (null without a fast path)
  LaunchFn launch_fast_streamk;  // the fast path's stream-K kernel (null without a fast path)
  // The fast path for transposed operands, by OperandLayout - 1 (null: not compiled for this tile).
  LaunchFn launch_transposed[3];
  LaunchFn launch_transposed_split[3];
  LaunchFn launch_general_split;  // the general tile's split-K kernel (null: not compiled for this tile)
  LaunchFn launch_plain;  // GemmTile in a kernel of its own: operands that no chunk of the general tile fits
};

template <class T, bool SPLIT = false, bool STREAMK = false>
hipError_t launch_tile(const KParams& p, int grid, hipStream_t stream) {
  hipLaunchKernelGGL((grouped_gemm_kernel<T, SPLIT, STREAMK>), dim3(grid), dim3(T::NT), 0, stream, p);
  return hipGetLastError();
}

// X-macro menus: X(E, BM, BN, BK, WAVES_M, WAVES_N, STAGES).  Each translation unit expands a
// menu into explicit kernel instantiations (device and host passes) and into the host table.
// The 8-wave 256x256 tiles with at least three stages run the ping-pong schedule
// (gemm_pingpong.h); every other 16-bit vector-layout tile runs FastTile's schedule.
template <class E, int BM, int BN, int BK, int WM, int WN, int S, int LAY = 0>
struct FastTileFor {
  using type = typename std::conditional<BM == 256 && BN == 256 && WM == 2 && WN == 4 && S >= 3,
                                         PingPongTile<E, BK, S, LAY>, FastTile<E, BM, BN, BK, WM, WN, S, LAY>>::type;
};
template <class E, int BM, int BN, int BK, int WM, int WN, int S, int LAY = 0>
using FastTileT = typename FastTileFor<E, BM, BN, BK, WM, WN, S, LAY>::type;
#define MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S) FastTileT<E, BM, BN, BK, WM, WN, S>
// The general kernel has no stage count; the wrapper keeps one instantiation per menu entry even
// when two entries differ only in the fast path's stages.
template <class E, int BM, int BN, int BK, int WM, int WN, int S, int PARTS>
struct GeneralTileEntry : GeneralTile<E, BM, BN, BK, WM, WN, PARTS> {};
#define MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S) GeneralTileEntry<E, BM, BN, BK, WM, WN, S, 1>
#define MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S) GeneralTileEntry<E, BM, BN, BK, WM, WN, S, 3>
#define MOEGEMM_GEN_TF32(E, BM, BN, BK, WM, WN, S) GeneralTileEntry<E, BM, BN, BK, WM, WN, S, 2>

// GemmTile's own kernels (inst_*_plain.hip), for launches none of whose operands the general tile can stage
// in chunks: beside that tile's loops GemmTile gets the larger tile's LDS and occupancy.
// [1024,2048]@[2048,1536] fp32 with every second column of A: 232 us in the general kernel, 141 in its own.
template <class E, int BM, int BN, int BK, int WM, int WN, int S>
struct PlainTileEntry : GemmTile<E, BM, BN, BK, WM, WN> {};
#define MOEGEMM_INST_PLAIN(E, BM, BN, BK, WM, WN, S)                                                                 \
  template __global__ void grouped_gemm_kernel<PlainTileEntry<E, BM, BN, BK, WM, WN, S>, false>(KParams);            \
  template hipError_t launch_tile<PlainTileEntry<E, BM, BN, BK, WM, WN, S>>(const KParams&, int, hipStream_t);
#define MOEGEMM_EXTERN_PLAIN(E, BM, BN, BK, WM, WN, S) \
  extern template hipError_t launch_tile<PlainTileEntry<E, BM, BN, BK, WM, WN, S>>(const KParams&, int, hipStream_t);

// fp32 launches: the input precision picks the kernel (three bf16 parts per operand, or TF32's two).
template <class IEEE, class TF32, bool SPLIT>
hipError_t launch_f32(const KParams& p, int grid, hipStream_t stream) {
  return p.tf32 ? launch_tile<TF32, SPLIT>(p, grid, stream) : launch_tile<IEEE, SPLIT>(p, grid, stream);
}

#define MOEGEMM_INST16(E, BM, BN, BK, WM, WN, S)                                                     \
  template __global__ void grouped_gemm_kernel<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S), false>(KParams); \
  template __global__ void grouped_gemm_kernel<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S), true>(KParams);
// The general kernels, in translation units of their own (inst_*_gen.hip) like the stream-K ones.
#define MOEGEMM_INST16_GEN(E, BM, BN, BK, WM, WN, S)                                                         \
  template __global__ void grouped_gemm_kernel<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S), false>(KParams);       \
  template hipError_t launch_tile<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S)>(const KParams&, int, hipStream_t);
// General tiles with a split-K kernel: one per size class, for the tuner to spread few tiles.
#define MOEGEMM_MENU_GEN_SPLIT(X, E)                                                                    \
  X(E, 256, 256, 32, 2, 4, 4) X(E, 128, 128, 64, 2, 2, 4) X(E, 128, 64, 64, 2, 2, 4)                    \
  X(E, 64, 128, 64, 2, 2, 4) X(E, 64, 64, 64, 2, 2, 4) X(E, 32, 128, 64, 1, 4, 4)                       \
  X(E, 16, 64, 128, 1, 4, 4)
#define MOEGEMM_INST16_GENSPLIT(E, BM, BN, BK, WM, WN, S)                                               \
  template __global__ void grouped_gemm_kernel<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S), true>(KParams);   \
  template hipError_t launch_tile<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S), true>(const KParams&, int, hipStream_t);
#define MOEGEMM_EXTERN16_GENSPLIT(E, BM, BN, BK, WM, WN, S) \
  extern template hipError_t launch_tile<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S), true>(const KParams&, int, hipStream_t);
#define MOEGEMM_MATCH_GENSPLIT(E, BM, BN, BK, WM, WN, S) \
  || (bm == BM && bn == BN && bk == BK && wm == WM && wn == WN && s == S)
constexpr bool general_split_compiled(int bm, int bn, int bk, int wm, int wn, int s) {
  return false MOEGEMM_MENU_GEN_SPLIT(MOEGEMM_MATCH_GENSPLIT, E);
}
template <class E, int BM, int BN, int BK, int WM, int WN, int S>
constexpr LaunchFn general_split_launch() {
  if constexpr (general_split_compiled(BM, BN, BK, WM, WN, S))
    return &launch_tile<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S), true>;
  else
    return nullptr;
}
#define MOEGEMM_EXTERN16_GEN(E, BM, BN, BK, WM, WN, S) \
  extern template hipError_t launch_tile<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S)>(const KParams&, int, hipStream_t);
// The stream-K kernels live in translation units of their own (inst_*_sk.hip): compiled next to
// the other kernels of a tile, their presence in the module changed the register allocation of
// those kernels (18 of 54 moved, one from 8 to 72 bytes of scratch).  Each such unit instantiates
// the kernel and its host launcher; the tables refer to the launchers through these declarations.
#define MOEGEMM_INST16_SK(E, BM, BN, BK, WM, WN, S)                                                        \
  template __global__ void grouped_gemm_kernel<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S), true, true>(KParams); \
  template hipError_t launch_tile<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S), true, true>(const KParams&, int,   \
                                                                                      hipStream_t);
#define MOEGEMM_EXTERN16_SK(E, BM, BN, BK, WM, WN, S)                                                          \
  extern template hipError_t launch_tile<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S), true, true>(const KParams&, int, \
                                                                                             hipStream_t);

// Transposed operands (OperandLayout): the tiles a caller's shapes need there, one table for the
// K-contiguous B of linear weights (prefill and decode tiles) and one for an M-contiguous A
// (weight gradients: long M and N, so only large and middle tiles), alone or with a K-contiguous
// B.  A tile outside these tables runs its general kernel on such operands.
#define MOEGEMM_MENU_BT(X, E)                                                                            \
  X(E, 256, 256, 32, 2, 4, 4, 2) X(E, 128, 256, 64, 2, 4, 3, 2) X(E, 128, 128, 64, 2, 2, 4, 2)           \
  X(E, 64, 256, 64, 1, 4, 3, 2) X(E, 64, 128, 64, 2, 2, 4, 2) X(E, 64, 64, 64, 2, 2, 4, 2)               \
  X(E, 32, 128, 64, 1, 4, 4, 2) X(E, 32, 128, 128, 1, 4, 3, 2) X(E, 16, 256, 64, 1, 4, 4, 2)             \
  X(E, 16, 128, 128, 1, 4, 4, 2) X(E, 16, 64, 128, 1, 4, 4, 2) X(E, 16, 64, 128, 1, 4, 7, 2)
#define MOEGEMM_MENU_AT(X, E)                                                                            \
  X(E, 256, 256, 32, 2, 4, 4, 1) X(E, 128, 256, 64, 2, 4, 3, 1) X(E, 128, 128, 64, 2, 2, 4, 1)           \
  X(E, 64, 128, 64, 2, 2, 4, 1) X(E, 64, 64, 64, 2, 2, 4, 1)                                             \
  X(E, 256, 256, 32, 2, 4, 4, 3) X(E, 128, 256, 64, 2, 4, 3, 3) X(E, 128, 128, 64, 2, 2, 4, 3)           \
  X(E, 64, 128, 64, 2, 2, 4, 3) X(E, 64, 64, 64, 2, 2, 4, 3)
#define MOEGEMM_INST16_TR(E, BM, BN, BK, WM, WN, S, LAY)                                                     \
  template __global__ void grouped_gemm_kernel<FastTileT<E, BM, BN, BK, WM, WN, S, LAY>, false>(KParams);    \
  template __global__ void grouped_gemm_kernel<FastTileT<E, BM, BN, BK, WM, WN, S, LAY>, true>(KParams);     \
  template hipError_t launch_tile<FastTileT<E, BM, BN, BK, WM, WN, S, LAY>, false>(const KParams&, int, hipStream_t); \
  template hipError_t launch_tile<FastTileT<E, BM, BN, BK, WM, WN, S, LAY>, true>(const KParams&, int, hipStream_t);
#define MOEGEMM_EXTERN16_TR(E, BM, BN, BK, WM, WN, S, LAY)                                                   \
  extern template hipError_t launch_tile<FastTileT<E, BM, BN, BK, WM, WN, S, LAY>, false>(const KParams&, int, \
                                                                                          hipStream_t);      \
  extern template hipError_t launch_tile<FastTileT<E, BM, BN, BK, WM, WN, S, LAY>, true>(const KParams&, int, \
                                                                                         hipStream_t);
#define MOEGEMM_MATCH_TR(E, BM, BN, BK, WM, WN, S, LAY) \
  || (bm == BM && bn == BN && bk == BK && wm == WM && wn == WN && s == S && lay == LAY)
constexpr bool transposed_compiled(int bm, int bn, int bk, int wm, int wn, int s, int lay) {
  return false MOEGEMM_MENU_BT(MOEGEMM_MATCH_TR, E) MOEGEMM_MENU_AT(MOEGEMM_MATCH_TR, E);
}
template <class E, int BM, int BN, int BK, int WM, int WN, int S, int LAY, bool SPLIT>
constexpr LaunchFn transposed_launch() {
  if constexpr (transposed_compiled(BM, BN, BK, WM, WN, S, LAY))
    return &launch_tile<FastTileT<E, BM, BN, BK, WM, WN, S, LAY>, SPLIT>;
  else
    return nullptr;
}
#define MOEGEMM_ENTRY16(E, BM, BN, BK, WM, WN, S)                                             \
  KernelEntry{E::dtype, BM, BN, BK, (WM) * (WN), S, WM, WN,                                   \
              MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S)::LDS_BYTES,                              \
              MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S)::SWIGLU_OK ? 1 : 0,                      \
              &launch_tile<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S)>,                          \
              &launch_tile<MOEGEMM_GEN(E, BM, BN, BK, WM, WN, S)>,                           \
              &launch_tile<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S), true>,                    \
              &launch_tile<MOEGEMM_FAST(E, BM, BN, BK, WM, WN, S), true, true>,              \
              {transposed_launch<E, BM, BN, BK, WM, WN, S, 1, false>(),                       \
               transposed_launch<E, BM, BN, BK, WM, WN, S, 2, false>(),                       \
               transposed_launch<E, BM, BN, BK, WM, WN, S, 3, false>()},                      \
              {transposed_launch<E, BM, BN, BK, WM, WN, S, 1, true>(),                        \
               transposed_launch<E, BM, BN, BK, WM, WN, S, 2, true>(),                        \
               transposed_launch<E, BM, BN, BK, WM, WN, S, 3, true>()},                       \
              general_split_launch<E, BM, BN, BK, WM, WN, S>(),                               \
              &launch_tile<PlainTileEntry<E, BM, BN, BK, WM, WN, S>>},

#define MOEGEMM_INST32(E, BM, BN, BK, WM, WN, S) \
  template __global__ void grouped_gemm_kernel<MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S), false>(KParams); \
  template __global__ void grouped_gemm_kernel<MOEGEMM_GEN_TF32(E, BM, BN, BK, WM, WN, S), false>(KParams);
#define MOEGEMM_INST32_SPLIT(E, BM, BN, BK, WM, WN, S) \
  template __global__ void grouped_gemm_kernel<MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S), true>(KParams); \
  template __global__ void grouped_gemm_kernel<MOEGEMM_GEN_TF32(E, BM, BN, BK, WM, WN, S), true>(KParams); \
  template hipError_t launch_f32<MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S), MOEGEMM_GEN_TF32(E, BM, BN, BK, WM, WN, S), \
                                 true>(const KParams&, int, hipStream_t);
#define MOEGEMM_EXTERN32_SPLIT(E, BM, BN, BK, WM, WN, S) \
  extern template hipError_t launch_f32<MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S), \
                                        MOEGEMM_GEN_TF32(E, BM, BN, BK, WM, WN, S), true>(const KParams&, int, hipStream_t);
#define MOEGEMM_ENTRY32(E, BM, BN, BK, WM, WN, S)                                             \
  KernelEntry{E::dtype, BM, BN, BK, (WM) * (WN), S, WM, WN,                                   \
              MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S)::LDS_BYTES, 0, nullptr,                    \
              &launch_f32<MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S), MOEGEMM_GEN_TF32(E, BM, BN, BK, WM, WN, S), false>, \
              nullptr, nullptr, {nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr},         \
              &launch_f32<MOEGEMM_GEN32(E, BM, BN, BK, WM, WN, S), MOEGEMM_GEN_TF32(E, BM, BN, BK, WM, WN, S), true>, \
              &launch_tile<PlainTileEntry<E, BM, BN, BK, WM, WN, S>>},

// 16-bit menu (bf16 and f16 share it): large-M MFMA-bound tiles down to skinny-M streaming tiles.
// STAGES is sized to the 160 KiB LDS of a CU; the 2-stage narrow tiles at the end fit two
// workgroups per CU (16x128 fits four; LDS, and registers via FastTile::WAVES_PER_EU), so one
// workgroup's prologue overlaps another's work on short-K groups.
// The 32x128 two- and three-stage tiles serve narrow groups of 17 to 32 rows: 128 experts of N = 384
// are 384 tiles of 128 columns, all resident at once (three workgroups a CU), where 256-column tiles
// left a half-empty second column tile per expert.  fp16 128 x [32,2048]@[2048,384], tuned: 49.9 us
// (4.4 TB/s) before, 41.9 us with them (5.3 TB/s); 64 x [32,4096]@[4096,512] 49.0 -> 47.1 us.
#define MOEGEMM_MENU_16BIT(X, E)                                                             \
  X(E, 256, 256, 64, 2, 4, 2) X(E, 256, 256, 64, 2, 2, 2) X(E, 256, 256, 32, 2, 2, 4)        \
  X(E, 256, 256, 32, 2, 4, 4)                                                                \
  X(E, 256, 128, 64, 2, 2, 3) X(E, 128, 256, 64, 2, 4, 3)                                   \
  X(E, 128, 256, 64, 2, 2, 3) X(E, 128, 128, 64, 2, 2, 4) X(E, 128, 64, 64, 2, 2, 4)         \
  X(E, 64, 256, 64, 1, 4, 3) X(E, 64, 128, 64, 2, 2, 4) X(E, 64, 64, 64, 2, 2, 4)            \
  X(E, 32, 256, 64, 1, 4, 4) X(E, 32, 128, 64, 1, 4, 4) X(E, 32, 128, 128, 1, 4, 3)          \
  X(E, 16, 256, 64, 1, 4, 4) X(E, 16, 256, 128, 1, 4, 2) X(E, 16, 128, 128, 1, 4, 4)         \
  X(E, 16, 64, 128, 1, 4, 4) X(E, 16, 64, 128, 1, 4, 7)                                    \
  X(E, 16, 256, 64, 1, 4, 2) X(E, 32, 256, 64, 1, 4, 2) X(E, 64, 128, 64, 2, 2, 2)        \
  X(E, 16, 128, 64, 1, 4, 2) X(E, 16, 512, 64, 1, 4, 2) X(E, 64, 512, 64, 1, 4, 2)        \
  X(E, 32, 512, 32, 1, 4, 4) X(E, 32, 128, 64, 1, 4, 2) X(E, 32, 128, 64, 1, 4, 3)

// fp32 menu (general kernel); STAGES is the register-staged double buffer.
#define MOEGEMM_MENU_F32(X, E)                                                               \
  X(E, 256, 128, 32, 4, 2, 2) X(E, 128, 128, 32, 2, 4, 2) X(E, 128, 128, 32, 2, 2, 2) X(E, 64, 64, 32, 2, 2, 2) X(E, 32, 64, 32, 1, 4, 2)            \
  X(E, 16, 64, 32, 1, 4, 2) X(E, 32, 32, 32, 1, 2, 2)

extern const KernelEntry kEntriesBf16[];
extern const int kNumBf16;
extern const KernelEntry kEntriesF16[];
extern const int kNumF16;
extern const KernelEntry kEntriesF32[];
extern const int kNumF32;

}  // namespace moegemm
