// Multi-token (prefill) projections on the bf16/f16 matrix cores of gfx950.
//
// Y[t][n] = sum_k X[t][k] * W[n][k] for a segment of M tokens and a raw GGUF
// weight matrix W (Q4_K, Q6_K or Q8_0). The product runs on
// v_mfma_f32_16x16x32_f16 (prefill.hip) or v_mfma_f32_32x32x16_f16
// (gemm_tiled.hip, gemm_q8.hip) with operands that make it exact up to fp32
// accumulation:
//  * W side: the integer quants times their integer sub-block scales, which
//    are small enough to be exact in f16 (Q4_K: q*sc <= 945; Q6_K: (q-32)*sc
//    split into 16*(q-32)*floor(sc/16) and (q-32)*(sc mod 16), in the tiled
//    kernel q - 32, its products scaled by d*sc in fp32; Q8_0: q); the fp16
//    block scales d (and dmin) are applied in fp32 once per block.
//  * X side: each token row scaled by a power of two s so that max|x*s| lies
//    in [2^14, 2^15), then split x*s = hi + lo into two f16 (22 significant
//    bits), both multiplied into the same accumulator.
// SplitRows prepares the X side once per segment (optionally fused with the
// RMSNorm that produces it); QGemm runs up to three weight matrices over it.
// Results satisfy the matvec row bound max|d|/sum|a*w| <= 1e-6 of the
// reference's own dot kernels (reference src/matmul.cc:73-124).

#ifndef RPG_HIP_PREFILL_H_
#define RPG_HIP_PREFILL_H_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "kernels.h"

namespace rpg {
namespace k {

// Device buffers of a split segment (M tokens, K inputs). Within every 8
// consecutive inputs the f16 copies are stored in the order 0,2,1,3,4,6,5,7
// (the order in which the weight operand is assembled from packed quants).
struct SplitX {
  void* hi = nullptr;      // f16 [M][K]
  void* lo = nullptr;      // f16 [M][K]
  void* sum_hi = nullptr;  // f16 [M][K/32]: sum of each 32 inputs * s/32, split
  void* sum_lo = nullptr;
  float* inv_s = nullptr;  // [M] 1/s
  // split-K partial products of QGemm: part_cap floats, of which the K-quants'
  // splits plan with part_floats, a function of the segment alone (a product's
  // order of sums follows its split)
  float* part = nullptr;
  int64_t part_floats = 0, part_cap = 0;
  int32_t M = 0, K = 0;
};
// Bytes of a SplitX for up to M x K whose QGemm launches produce at most
// n_max output columns in total (sizes the split-K partials); q8: Q8_0
// matrices among them.
size_t SplitXBytes(int M, int K, int n_max, bool q8);
// Carve a SplitX out of `base` (SplitXBytes of the same figures).
SplitX SplitXView(void* base, int M, int K, int n_max, bool q8);

// x = X rows (stride ldx), or RMSNorm(x) * norm_w when norm_w != nullptr
// (double sum of squares, float scale, (x * scale) * w, reference
// src/kernels.h:56-63).
void SplitRows(const float* X, int64_t ldx, int M, int K, const float* norm_w, float eps, const SplitX& out,
               hipStream_t s);

// SplitRows over X after adding the pending sums to X (written back: X is
// the residual stream), the bits of the reduce launch followed by SplitRows.
void SplitRowsAdd(float* X, int64_t ldx, int M, int K, const float* norm_w, float eps, const SplitX& out,
                  const SplitPending& pend, hipStream_t s);
// The reduce launch of a pending sum, added to or stored in y (row stride ldy,
// N columns).
void ApplyPending(const SplitPending& pend, float* y, int64_t ldy, int N, hipStream_t s, Epilogue epi = kAdd);

// Compute units of the current device (queried once per device).
int ComputeUnits();

struct GemmJob {
  MatRef w;
  float* y = nullptr;
  int64_t ldy = 0;
  Epilogue epi = kStore;
};
// True when W can run on QGemm (K-quants need K a multiple of 256).
bool QGemmSupports(const MatRef& w);
// Jobs of one launch have one type.
void QGemm(const SplitX& x, const GemmJob* jobs, int n_jobs, hipStream_t s, SplitPending* defer = nullptr);
// (defer: one entry per job; a K split's sums are left to the caller, to add
// or store before y is read -- SplitRowsAdd, QkNormRopeCache, ApplyPending.
// defer[j].part stays null when nothing is pending)
// gate.y[t][r] = silu(gate row r . x_t) * (up row r . x_t) in one launch,
// the same bits as two QGemm products and SwiGLURows -- except where a tiled
// launch runs its last round's tiles in K parts (Q4_K: halves, where that round
// is at most half full): those rows' sums are the parts' sums added, within
// the products' row bound. Q4_K or Q8_0 gate and up of one shape; for Q4_K only
// where QGemm would not split K. False (nothing launched) otherwise.
bool QGemmSwiGLU(const SplitX& x, const GemmJob& gate, const GemmJob& up, hipStream_t s);

// y[i] = silu(g[i]) * u[i] (reference src/kernels.h:82-92), n elements.
void SwiGLURows(const float* g, const float* u, float* y, int64_t n, hipStream_t s);

// Tiled Q4_K / Q6_K GEMM (gemm_tiled.hip): 128 tokens x 128 weight rows per
// workgroup, each step's weights unpacked once into LDS. QGemm and QGemmSwiGLU
// take it for segments of at least kTiledMinTokens tokens.
// The form of gemm_q8.hip (64 x 64 wave tiles, weights unpacked in registers)
// was faster for these too (4B 512 tokens 14.1 -> 12.7 ms) and closer to
// float64, but another order of sums gives another reply to a seed wherever a
// draw falls between two roundings.
constexpr int kTiledTokens = 128;
constexpr int kTiledRows = 128;
constexpr int kTiledMinTokens = 96;

struct TiledArgs {
  SplitX x;
  GemmJob job[3];
  int32_t tiles[3];  // 128-row tiles per job (pair: 64-row tiles of gate and up)
  int32_t n_jobs;
  int32_t tiles_m;   // 128-token tiles; workgroup i takes token tile i % tiles_m
  int32_t ksplit;    // blockIdx.y takes super-blocks [y * n / ksplit, (y + 1) * n / ksplit)
  int64_t part_ld;   // partials: x.part[(z * M + token) * part_ld + pcol[job] + row]
  int32_t pcol[3];
  int32_t pair;      // job 0 gate, job 1 up: y = silu(gate.x) * (up.x), no K split
  // pair only, 0 = none: workgroups from tail_wg on take the tiles from
  // tail_wg on in halves (the two super-block halves of each, raw sums to
  // x.part, kTiledTailFloats per half), finished by a second launch
  int32_t tail_wg = 0;
};
constexpr int kTiledTailFloats = kTiledTokens * kTiledRows;
void LaunchTiled(const TiledArgs& a, hipStream_t s);

// Tiled Q8_0 GEMM (gemm_q8.hip; K a multiple of 256): 64 or 128 tokens x 256
// weight rows per workgroup. Tiles of 64 tokens fill the compute units with
// fewer K parts and pad less; from about 320 tokens on the 128-token tiles'
// fewer LDS bytes per product win (measured on the kernel's Q4_K form, a
// segment behind 600 tokens, ms, 64 / 128-token tiles: 1.7B 65 tokens 4.7 / 5.9,
// 300 6.2 / 7.5, 512 8.7 / 8.8).
constexpr int kQ8Rows = 256;
inline int Q8TileTokens(int M) { return M <= 320 ? 64 : 128; }

struct Q8TiledArgs {
  SplitX x;
  GemmJob job[3];
  int32_t tiles[3];  // 256-row tiles per job (pair: 128-row tiles of gate and up)
  int32_t n_jobs;
  int32_t tokens;    // Q8TileTokens(x.M)
  int32_t tiles_m;   // token tiles; workgroup i takes token tile i % tiles_m
  int32_t ksplit;    // blockIdx.y takes super-blocks [y * n / ksplit, (y + 1) * n / ksplit)
  int64_t part_ld;   // partials: x.part[(z * M + token) * part_ld + pcol[job] + row]
  int32_t pcol[3];
  int32_t pair;      // job 0 gate, job 1 up: y = silu(gate.x) * (up.x), no K split
  // pair only, tail_split > 1: the tiles from tail_wg on run as tail_split K
  // parts each (raw sums to x.part, tokens x kQ8Rows floats per part), finished
  // by a second launch
  int32_t tail_wg = 0, tail_split = 1;
};
void LaunchQ8Tiled(const Q8TiledArgs& a, hipStream_t s);

}  // namespace k
}  // namespace rpg

#endif  // RPG_HIP_PREFILL_H_
