// Tiled prefill GEMM of Q8_0 weights: v_mfma_f32_32x32x16_f16 over 64 or 128
// tokens x 256 rows, for segments of every length past the few-token matvec.
//
// The operands are those of prefill.h (the int8 quants exact in f16, token
// rows split into f16 hi + lo, the fp16 block scales applied in fp32), so
// every output meets the same bound as QGemm8Kernel's. What differs is where
// the work sits:
//  * each of the 8 waves owns 64 tokens x 64 rows (2 x 2 tiles; 64 x 32 in a
//    tile of 64 tokens): per step of 64 inputs it reads 16 KB of token
//    operands and 4 KB of raw quants from LDS for 32 products, and unpacks its
//    own weight operands in registers, each for four products (two token
//    tiles, hi and lo);
//  * the tokens' hi/lo rows of the step arrive by LDS DMA; the raw quants
//    pass through a register ring, so any block alignment is served;
//  * a block's sums are scaled into the fp32 sums as the next block's products
//    run;
//  * the epilogue takes the token scales from LDS: loaded there one by one,
//    each load waited for the stores before it (15 us of a 42 us launch).
// One workgroup per compute unit (two waves per SIMD).
//
// What bounds it: with every compute unit at work the card lowers its clock
// -- the loop without loads or unpacking takes 0.98 us per step on 128
// compute units and 1.66 us on 256 (1.29 PFLOP/s issued, half of it useful:
// hi and lo); this loop takes 1.8 us. A library f16 product of 4096^3 random
// values reaches 1.07 - 1.2 PFLOP/s on the same card. Short launches pay
// ~7 us of launch, pipeline fill and output besides. Measured, the 1.7B Q8_0
// prefill of 777 tokens: 23.1 ms on QGemm8Kernel, 10.3 ms here.
//
// MFMA layout (gfx950): 32x32x16 f16: lane l holds A[l % 32][8 (l / 32) ..
// +8) and B[8 (l / 32) .. +8][l % 32]; the 16 results of lane l are
// C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32], v < 16.

#include <hip/hip_runtime.h>

#include "common.h"
#include "expf_glibc.h"
#include "prefill.h"
#include "quant_dev.h"

namespace rpg {
namespace k {

namespace {

typedef _Float16 H2 __attribute__((ext_vector_type(2)));
typedef _Float16 H8 __attribute__((ext_vector_type(8)));
typedef float F16v __attribute__((ext_vector_type(16)));
typedef uint32_t U2 __attribute__((ext_vector_type(2)));
typedef uint32_t U4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;    // 8 waves
constexpr int kTN = kQ8Rows;     // weight rows per workgroup

// 16 bytes at an address that is only 2-byte aligned (Q8_0 blocks are 34 bytes
// long): one dwordx4 load, which global memory serves at any byte alignment.
typedef U4 U4A2 __attribute__((aligned(2)));

template <typename T>
__device__ __forceinline__ T GLoad(const void* p) {
  return *(const __attribute__((address_space(1))) T*)(p);
}

typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc MakeRsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
}

// 16 bytes per lane from the resource to LDS (a wave's lanes side by side).
__device__ __forceinline__ void DmaLds(Rsrc src, void* lds, uint32_t voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)lds, 16, voff, soff, 0, 0);
}

// Chunk swizzle of the token rows in LDS (128-byte rows, 16-byte chunks):
// logical chunk c of row r sits at chunk c ^ ASwz(r). Any 8 consecutive rows
// (from a multiple of 8) use 8 different chunks, and so do the 8 even and the
// 8 odd rows of any 16, so the b128 reads of 32 consecutive rows at one
// logical chunk meet no bank conflict with either 32 or 64 banks.
__device__ __forceinline__ int ASwz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

__device__ __forceinline__ uint32_t AsU(H2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ H2 AsH2(uint32_t v) { return __builtin_bit_cast(H2, v); }

__device__ __forceinline__ F16v Mma(H8 a, H8 b, F16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
// A product from zero. The empty asm after it marks both sources as still in
// use, so the result is never allocated over them: an MFMA whose destination
// aliases its A or B registers returned wrong sums on gfx950 (measured), and
// the compiler allows that allocation when a source dies at the product.
__device__ __forceinline__ F16v MmaFresh(H8 a, H8 b) {
  const F16v r = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, F16v{}, 0, 0, 0);
  asm volatile("" ::"v"(a), "v"(b), "v"(r));
  return r;
}
// Keeps the computation of t at its place.
__device__ __forceinline__ void Pin(F16v& t) { asm volatile("" : "+v"(t)); }

// Weight operands of 8 inputs (two dwords of bytes), in the operand order of
// SplitX (within every 8 inputs: 0, 2, 1, 3, 4, 6, 5, 7): bytes u = q + 128
// read as the f16 1024 + u, less 1152: the exact q, negated if neg.
__device__ __forceinline__ H8 UnpackBytes(uint32_t v0, uint32_t v1, uint32_t magic, bool neg) {
  const H2 off = H2{static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)};
  const H2 v[4] = {AsH2(__builtin_amdgcn_perm(magic, v0, 0x04020400u)),
                   AsH2(__builtin_amdgcn_perm(magic, v0, 0x04030401u)),
                   AsH2(__builtin_amdgcn_perm(magic, v1, 0x04020400u)),
                   AsH2(__builtin_amdgcn_perm(magic, v1, 0x04030401u))};
  U4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = AsU(neg ? off - v[i] : v[i] - off);
  return __builtin_bit_cast(H8, r);
}

// A step is two 32-weight blocks of a super-block of 256 inputs (the unit of
// the K split).
//
// kTM: tokens per workgroup. 128: waves in 2 token halves x 4 row quarters,
// each 64 tokens x 64 rows; 64: 8 row eighths, each 64 tokens x 32 rows.
template <int kTM>
struct TileLds {
  // quants of a step, 16-byte chunks side by side over the rows (a wave's
  // reads of one chunk are 512 consecutive bytes): [stage][2 p + h][row]:
  // unsigned bytes, inputs 8 h .. + 8 of slices 2 p and 2 p + 1 (slice: 16
  // inputs of the step)
  U4 Bq[2][4][kTN];
  alignas(16) float Sc[2][kTN][2];  // [stage][row]: d of its 2 blocks
  alignas(16) float Is[kTM];        // 1 / s of the token rows
};

// Part zt of the tile's K (zt < 0: this launch's part blockIdx.y), tile (tm,
// nt) of job j. As0, As1: a stage's token rows [hi, lo][token] each, swizzled
// (ASwz): one array per stage, since the compiler tells LDS arrays apart when
// it places the waits for its DMA loads, so that reads of one stage do not
// wait for the DMA into the other.
template <int kTM>
__device__ __forceinline__ void Q8Tile(const Q8TiledArgs& a, int wgi, int zt, int tm, int nt, int j,
                                       _Float16 (&As0)[2][kTM][64], _Float16 (&As1)[2][kTM][64], TileLds<kTM>& L) {
  constexpr int kNI = kTM / 64;    // 32-row tiles per wave
  constexpr int kWN = 32 * kNI;    // rows per wave
  constexpr int kDma = kTM / 32;   // DMA loads of a step's token rows per wave
  const int ts = a.tail_split;
  const GemmJob& J = a.job[j];
  const SplitX& x = a.x;
  const int M = x.M, K = x.K;
  // this part's super-blocks [o0, o1)
  const int z = blockIdx.y, nall = K >> 8;
  const int o0 = zt >= 0 ? zt * nall / ts : z * nall / a.ksplit;
  const int o1 = zt >= 0 ? (zt + 1) * nall / ts : (z + 1) * nall / a.ksplit;
  const int m0 = tm * kTM;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = kNI == 2 ? wave >> 2 : 0, wn = kNI == 2 ? wave & 3 : wave;  // 64-token half, kWN rows
  const int l32 = lane & 31, lh = lane >> 5;
  const int rows = J.w.rows;
  const int64_t rb = J.w.row_bytes;
  const bool pair = a.pair != 0;

  // Two stages (a step's operands) alternate.
  auto as = [&](int st) -> _Float16(*)[kTM][64] { return st ? As1 : As0; };
  auto& Bq = L.Bq;
  auto& Sc = L.Sc;
  auto& Is = L.Is;

  // The weight row this thread stages, as local row br, and the block bq of a
  // step (slices 2 bq and 2 bq + 1). A pair's workgroup holds 128 output rows;
  // even waves stage gate rows, odd ones up rows (the matrix is wave-uniform).
  // A wave's rows are gate rows and then the same up rows: 32 + 32 as its two
  // tiles, or 16 + 16 of its one.
  const int bq = tid & 1, bi = (tid >> 1) & 31;
  const int pr = 32 * (wave >> 1) + bi;  // (pair: row of the 128)
  const int br = kNI == 1 && pair ? 32 * (pr >> 4) + 16 * (wave & 1) + (pr & 15) : tid >> 1;
  const uint8_t* bmat = (pair && (wave & 1)) ? a.job[1].w.w : J.w.w;
  const int brow_i = pair ? min(128 * nt + pr, rows - 1) : min(kTN * nt + br, rows - 1);
  // (2-byte aligned global loads, a uniform base and a 32-bit lane offset)
  const uint32_t b_lane = static_cast<uint32_t>(brow_i) * static_cast<uint32_t>(rb) + 34u * bq;
  // The token rows of a step reach LDS by DMA (buffer loads with an LDS
  // destination: a wave's 64 lanes x 16 bytes land as 1 KB in a row). A
  // step's rows are 2 parts x kTM tokens x 128 bytes = kTM / 4 such loads,
  // kDma per wave: load i of wave w fills part w / 4, rows 8 b .. 8 b + 7, b =
  // (kDma w + i) % (kTM / 8); lane L reads token row 8 b + L / 8 and lands at chunk
  // L % 8 of it, which holds logical chunk (L % 8) ^ ASwz(row): step inputs
  // 8 c .. + 8. The buffer resources end at the last token, so the rows past
  // it read as zeros.
  const uint32_t a_bytes = static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 2u;
  const Rsrc ra_src = MakeRsrc(wave < 4 ? x.hi : x.lo, a_bytes);
  uint32_t a_voff[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = 8 * ((kDma * wave + i) & (kTM / 8 - 1)) + (lane >> 3);
    const int lc = (lane & 7) ^ ASwz(r);
    a_voff[i] = (static_cast<uint32_t>(m0 + r) * static_cast<uint32_t>(K) + 8u * lc) * 2u;
  }

  const uint32_t magic8 = 0x64646464u;

  // The weights' loads run kAhead steps ahead in a register ring: step g's
  // quant bytes and scale sit in slot g % kSlots from their issue until they
  // are staged. Every step issues the same loads, unconditionally (steps past
  // the end re-read the last one), so the compiler counts them and waits for
  // one step's loads while the next steps' stay in flight.
  constexpr int kAhead = 3, kSlots = kAhead - 1;
  U4 rl[kSlots], rh[kSlots];
  uint32_t rd[kSlots];
  const int nsteps = 4 * (o1 - o0);
  // VMEM instructions of one issue() (fewer would only wait longer, more would
  // let a step read rows still in flight)
  constexpr int kLoads = 3;
  // the token rows of step g (g = 4 o + s of this part, super-block o0 + o)
  // into stage st
  auto issue_a = [&](int g, int st) {
    g = min(g, nsteps - 1);
    const int ob = o0 + (g >> 2), s = g & 3;
    const int so = 2 * (256 * ob + 64 * s);
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      DmaLds(ra_src, &as(st)[wave >> 2][8 * ((kDma * wave + i) & (kTM / 8 - 1))][0], a_voff[i], so);
  };
  auto issue = [&](int g, int slot) {
    g = min(g, nsteps - 1);
    const uint8_t* blk = bmat + 34 * static_cast<int64_t>(8 * (o0 + (g >> 2)) + 2 * (g & 3));
    rl[slot] = GLoad<U4A2>(blk + 2 + b_lane);
    rh[slot] = GLoad<U4A2>(blk + 18 + b_lane);
    rd[slot] = GLoad<uint16_t>(blk + b_lane);
  };
  // the quants and scales of a step into stage st
  auto store_b = [&](int slot, int st) {
    const uint32_t f = 0x80808080u;
    const U4 q0 = rl[slot], q1 = rh[slot];
    Bq[st][2 * bq][br] = U4{q0.x ^ f, q0.y ^ f, q1.x ^ f, q1.y ^ f};
    Bq[st][2 * bq + 1][br] = U4{q0.z ^ f, q0.w ^ f, q1.z ^ f, q1.w ^ f};
    Sc[st][br][bq] = dev::HalfToFloatFast(rd[slot]);
  };

  // A block's products accumulate in P from zero and are scaled into T while
  // the next block's run (the first time that adds zeros): its two slices
  // multiply the tokens' lo parts, then the hi parts (lo products added to
  // sums of the hi parts' size round at that size, which over long chains
  // measured two to three times the error).
  // The matrix core rounds its sums down (measured: a common negative error
  // of every token, which an attention average keeps where it averages the
  // tokens' own errors out), so every odd block multiplies the negated
  // weights and is subtracted: the two halves' errors cancel.
  F16v T[2][kNI], P[2][kNI];
  float Cs[kNI] = {};
#pragma unroll
  for (int i = 0; i < 2 * kNI; ++i) {
    T[i / kNI][i % kNI] = F16v{};
    P[i / kNI][i % kNI] = F16v{};
  }

  // token operands of one slice and part, double-buffered; the weight
  // operands of a block; the quants of the wave's rows (slices 2 p and 2 p +
  // 1) and their scales
  H8 op[2][2], b[2][kNI];
  U4 qv[kNI];
  float sc[kNI];
  auto read_a = [&](H8* q, int st, int part, int kk) {
    const int lc = 2 * kk + lh;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
      const int ar = 64 * wm + 32 * mi + l32;
      q[mi] = *reinterpret_cast<const H8*>(&as(st)[part][ar][8 * (lc ^ ASwz(ar))]);
    }
  };
  auto read_q = [&](int st, int p) {
#pragma unroll
    for (int ni = 0; ni < kNI; ++ni) {
      const int r = kWN * wn + 32 * ni + l32;
      qv[ni] = Bq[st][2 * p + lh][r];
      sc[ni] = Sc[st][r][p];
    }
  };

  // (read again by the epilogue from LDS: loads there would wait for its
  // stores)
  if (tid < kTM) Is[tid] = x.inv_s[min(m0 + tid, M - 1)];
  // prologue: step 0 staged, step 1's token rows and weights and step 2's
  // weights in flight
  issue_a(0, 0);
  issue(0, 0);
  issue(1, 1);
  store_b(0, 0);
  issue(2, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  issue_a(1, 1);
  read_a(op[0], 0, 1, 0);
  read_q(0, 0);
  for (int o = 0; o < o1 - o0; ++o) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      // step g = 4 o + s multiplies stage s % 2 while step g + 1's weights are
      // staged into the other one, where its token rows' DMA, issued a step
      // ago, lands. The barrier sits before the last of the step's 8 items (a
      // slice and part), whose operands are in registers by then: past it the
      // next step's first operands are read while that item multiplies, and
      // step g + 2's DMA is issued.
      const int g = 4 * o + s, st = s & 1, nx = st ^ 1, ns = (s + 1) & 3;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int kk = ((i >> 2) << 1) | (i & 1), hi = (i >> 1) & 1, kg = kk & 1;
        if (i == 7) {
          // step g + 1's token rows have landed (only the weight loads issued
          // in this step, after them, may still be in flight)
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
          __syncthreads();
          read_a(op[0], nx, 1, 0);
        } else {
          const int k1 = (((i + 1) >> 2) << 1) | ((i + 1) & 1), h1 = ((i + 1) >> 1) & 1;
          read_a(op[(i + 1) & 1], st, h1 ^ 1, k1);
        }
        if (!hi) {
#pragma unroll
          for (int ni = 0; ni < kNI; ++ni)
            b[kg][ni] = UnpackBytes(qv[ni][2 * kg], qv[ni][2 * kg + 1], magic8, kk >> 1);
        }
        const H8* q = op[i & 1];
        const bool fresh = !hi && kg == 0;
        const bool last_neg = kk >> 1 == 0;  // P's block was an odd one
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
          for (int ni = 0; ni < kNI; ++ni) {
            if (fresh) {
#pragma unroll
              for (int v = 0; v < 16; ++v)
                T[mi][ni][v] = __builtin_fmaf(last_neg ? -Cs[ni] : Cs[ni], P[mi][ni][v], T[mi][ni][v]);
              // (here, not later: the compiler would else keep both P)
              Pin(T[mi][ni]);
              P[mi][ni] = MmaFresh(q[mi], b[kg][ni]);
              __builtin_amdgcn_sched_barrier(0);  // (a tile's sums scaled, then overwritten)
            } else {
              P[mi][ni] = Mma(q[mi], b[kg][ni], P[mi][ni]);
            }
          }
        if (fresh) {
#pragma unroll
          for (int ni = 0; ni < kNI; ++ni) Cs[ni] = sc[ni];
        }
        // the next step's staging, spread over the items
        if (i == 3) read_q(st, 1);
        if (i == 3) store_b(ns % kSlots, nx);
        if (i == 4) issue(g + kAhead, ns % kSlots);
        if (i == 7) {
          read_q(nx, 0);
          // (the DMA after these reads, which the compiler would else make
          // wait for it)
          __builtin_amdgcn_sched_barrier(0);
          issue_a(g + 2, st);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // epilogue: result v of tile (mi, ni) is token 64 wm + 32 mi + 8 (v / 4) +
  // 4 lh + v % 4, local row kWN wn + 32 ni + l32
  constexpr int kHalf = kWN / 2;  // a pair: gate rows of the wave, then its up rows
#pragma unroll
  for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
    for (int ni = 0; ni < kNI; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) T[mi][ni][v] = __builtin_fmaf(-Cs[ni], P[mi][ni][v], T[mi][ni][v]);  // (an odd one)
    // a quad of tokens at a time: 8 (v / 4) + 4 lh + [0, 4)
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4) {
      const int t0 = 64 * wm + 32 * mi + 8 * v4 + 4 * lh;
      const float4 is4 = *reinterpret_cast<const float4*>(&Is[t0]);
      const float is[4] = {is4.x, is4.y, is4.z, is4.w};
      if (zt >= 0) {
        // a part of a tail tile: raw sums, [token][local row]
        float* pt = x.part + (static_cast<int64_t>(wgi - a.tail_wg) * ts + zt) * (kTM * kTN) + t0 * kTN + kWN * wn + l32;
#pragma unroll
        for (int ni = 0; ni < kNI; ++ni)
#pragma unroll
          for (int e = 0; e < 4; ++e) pt[e * kTN + 32 * ni] = T[mi][ni][4 * v4 + e];
      } else if (pair) {
        // gate and up of the same row -- tiles 0 and 1, or lanes l32 and l32 +
        // 16 of the one tile: silu(g) * u (reference src/kernels.h:82-92), the
        // bits of the unfused stores followed by SwiGLURows
        const int row = 128 * nt + kHalf * wn + l32 % kHalf;
        float* y = J.y + static_cast<int64_t>(m0 + t0) * J.ldy + row;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float tg = T[mi][0][4 * v4 + e];
          float tu;
          if constexpr (kNI == 2)
            tu = T[mi][kNI - 1][4 * v4 + e];
          else
            tu = __shfl_xor(tg, 16, 64);
          const float g = tg * is[e], u = tu * is[e];
          const float sg = g / __fadd_rn(1.0f, GlibcExpf(-g));
          if (row < rows && m0 + t0 + e < M && l32 < kHalf) y[e * J.ldy] = __fmul_rn(sg, u);
        }
      } else {
#pragma unroll
        for (int ni = 0; ni < kNI; ++ni) {
          const int row = kTN * nt + kWN * wn + 32 * ni + l32;
          float val[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) val[e] = T[mi][ni][4 * v4 + e] * is[e];
          if (row >= rows) continue;
          if (a.ksplit > 1) {
            float* pt = x.part + (static_cast<int64_t>(z) * M + m0 + t0) * a.part_ld + a.pcol[j] + row;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (m0 + t0 + e < M) pt[e * a.part_ld] = val[e];
          } else {
            float* y = J.y + static_cast<int64_t>(m0 + t0) * J.ldy + row;
            if (J.epi == kAdd) {
              float y0[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) y0[e] = m0 + t0 + e < M ? y[e * J.ldy] : 0.0f;
#pragma unroll
              for (int e = 0; e < 4; ++e) val[e] = y0[e] + val[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (m0 + t0 + e < M) y[e * J.ldy] = val[e];
          }
        }
      }
    }
  }
}

template <int kTM>
__global__ __launch_bounds__(kThreads) void Q8GemmKernel(Q8TiledArgs a) {
  __shared__ __align__(16) _Float16 As0[2][kTM][64];
  __shared__ __align__(16) _Float16 As1[2][kTM][64];
  __shared__ TileLds<kTM> L;
  // the tiles from tail_wg on in K parts: workgroup tail_wg + ts i + z takes
  // part z of tile tail_wg + i
  int wgi = static_cast<int>(blockIdx.x), zt = -1;
  const int ts = a.tail_split;
  if (ts > 1 && wgi >= a.tail_wg) {
    const int u = wgi - a.tail_wg;
    wgi = u / ts;
    zt = u - wgi * ts;
    wgi += a.tail_wg;
  }
  const int tm = wgi % a.tiles_m;
  int nt = wgi / a.tiles_m, j = 0;
  while (j + 1 < a.n_jobs && nt >= a.tiles[j]) {
    nt -= a.tiles[j];
    ++j;
  }
  Q8Tile<kTM>(a, wgi, zt, tm, nt, j, As0, As1, L);
}

// The tail tiles of a pair launch: y = silu(g) * u with g, u the sums of the
// tile's K parts (added in part order, then scaled as the full tiles' sums
// are), the full tiles' SwiGLU arithmetic. Workgroup (tile, y) takes tokens
// 8 y .. 8 y + 7 of the tile, four outputs per thread.
constexpr int kTailPer = 4;
template <int kTM>
__global__ __launch_bounds__(256) void TailSwiGLUKernel(Q8TiledArgs a) {
  constexpr int kHalf = 16 * (kTM / 64);  // a wave's gate rows, followed by its up rows
  const int tt = static_cast<int>(blockIdx.x), tile = a.tail_wg + tt;
  const int tm = tile % a.tiles_m, nt = tile / a.tiles_m;
  const GemmJob& J = a.job[0];
  const int rows = J.w.rows, M = a.x.M;
  const float* p = a.x.part + static_cast<int64_t>(tt) * a.tail_split * (kTM * kTN);
  float g[kTailPer], u[kTailPer], is[kTailPer];
#pragma unroll
  for (int i = 0; i < kTailPer; ++i) {
    const int e = (static_cast<int>(blockIdx.y) * kTailPer + i) * 256 + static_cast<int>(threadIdx.x);
    const int tl = e >> 7, c = e & 127;
    // (tokens past M: their sums, of zero rows, are read but not used)
    const float* q = p + tl * kTN + 2 * kHalf * (c / kHalf) + c % kHalf;
    g[i] = q[0];
    u[i] = q[kHalf];
    is[i] = a.x.inv_s[min(tm * kTM + tl, M - 1)];
  }
  for (int z = 1; z < a.tail_split; ++z) {
#pragma unroll
    for (int i = 0; i < kTailPer; ++i) {
      const int e = (static_cast<int>(blockIdx.y) * kTailPer + i) * 256 + static_cast<int>(threadIdx.x);
      const int tl = e >> 7, c = e & 127;
      const float* q = p + static_cast<int64_t>(z) * (kTM * kTN) + tl * kTN + 2 * kHalf * (c / kHalf) + c % kHalf;
      g[i] += q[0];
      u[i] += q[kHalf];
    }
  }
#pragma unroll
  for (int i = 0; i < kTailPer; ++i) {
    const int e = (static_cast<int>(blockIdx.y) * kTailPer + i) * 256 + static_cast<int>(threadIdx.x);
    const int tl = e >> 7, c = e & 127;
    const int tok = tm * kTM + tl, row = 128 * nt + c;
    if (tok >= M || row >= rows) continue;
    const float gv = g[i] * is[i], uv = u[i] * is[i];
    const float sg = gv / __fadd_rn(1.0f, GlibcExpf(-gv));
    J.y[static_cast<int64_t>(tok) * J.ldy + row] = __fmul_rn(sg, uv);
  }
}

}  // namespace

void LaunchQ8Tiled(const Q8TiledArgs& a, hipStream_t s) {
  int tiles = 0;
  for (int j = 0; j < a.n_jobs; ++j) tiles += a.tiles[j];
  for (int j = 0; j < a.n_jobs + (a.pair ? 1 : 0); ++j)
    RPG_CHECK(a.job[j].w.type == kQ8_0, "q8 gemm: weight type %u", a.job[j].w.type);
  RPG_CHECK(a.x.K % 256 == 0 && a.x.K >= 256, "q8 gemm: K = %d is not a multiple of 256", a.x.K);
  RPG_CHECK(a.tokens == Q8TileTokens(a.x.M) && a.tiles_m == CeilDiv(a.x.M, a.tokens), "q8 gemm: bad token tiles");
  RPG_CHECK(a.ksplit >= 1 && a.ksplit <= a.x.K / 256, "q8 gemm: bad K split %d", a.ksplit);
  const int total = tiles * a.tiles_m;
  const int n_tail = a.tail_split > 1 ? total - a.tail_wg : 0;
  if (a.tail_split > 1)
    RPG_CHECK(a.pair && a.ksplit == 1 && a.tail_wg >= 0 && a.tail_wg < total && a.tail_split <= a.x.K / 256 &&
                  static_cast<int64_t>(n_tail) * a.tail_split * a.tokens * kTN <= a.x.part_cap,
              "q8 gemm: bad tail split %d from workgroup %d of %d", a.tail_split, a.tail_wg, total);
  const dim3 grid(static_cast<unsigned>(total + n_tail * (a.tail_split - 1)), static_cast<unsigned>(a.ksplit));
  const bool small = a.tokens == 64;
  if (small)
    hipLaunchKernelGGL(Q8GemmKernel<64>, grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL(Q8GemmKernel<128>, grid, dim3(kThreads), 0, s, a);
  HIP_CHECK(hipGetLastError());
  if (n_tail > 0) {
    const dim3 tail_grid(static_cast<unsigned>(n_tail), static_cast<unsigned>(a.tokens * (kTN / 2) / (256 * kTailPer)));
    if (small)
      hipLaunchKernelGGL(TailSwiGLUKernel<64>, tail_grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL(TailSwiGLUKernel<128>, tail_grid, dim3(256), 0, s, a);
    HIP_CHECK(hipGetLastError());
  }
}

}  // namespace k
}  // namespace rpg
