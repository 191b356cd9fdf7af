// Tiled prefill GEMM for long segments: Q4_K, Q6_K and Q8_0 weights,
// v_mfma_f32_32x32x16_f16 over 128 tokens x 256 rows.
//
// The operands are those of prefill.h (exact integer weight operands, token
// rows split into f16 hi + lo, the fp16 block scales applied in fp32), so
// every output meets the same bound. What differs from the 32-token kernels
// is where the work sits:
//  * each of the 8 waves owns 64 tokens x 64 rows (2 x 2 tiles): per step of
//    64 inputs it reads 16 KB of token operands and 2 - 4 KB of raw quants
//    from LDS for 32 products, and unpacks its own weight operands in
//    registers, each for four products (two token tiles, hi and lo). A tile
//    of 32 tokens x 64 rows per wave, the weights unpacked once per workgroup
//    into LDS as f16, moved 176 KB of LDS per step for half the products;
//  * the tokens' hi/lo rows of the step arrive by LDS DMA; the raw quants
//    pass through a register ring, so any block alignment is served;
//  * scale groups (Q4_K: a step, the sub-block scales folded into the exact
//    operands; Q8_0: a block; Q6_K: a sub-block) are scaled into the fp32
//    sums as the next group's products run;
//  * Q4_K: the min term sum_j m_j * sum(x in sub-block j) of a super-block
//    is one v_mfma_f32_32x32x16_f16 over the 8 hi and 8 lo sub-block sums;
//  * the epilogue takes the token scales from LDS: loaded there one by one,
//    each load waited for the stores before it (15 us of a 42 us launch).
// One workgroup per compute unit (two waves per SIMD).
//
// What bounds it: with every compute unit at work the card lowers its clock
// -- the loop without loads or unpacking takes 0.98 us per step on 128
// compute units and 1.66 us on 256 (1.29 PFLOP/s issued, half of it useful:
// hi and lo); this loop takes 1.8 us. A library f16 product of 4096^3 random
// values reaches 1.07 - 1.2 PFLOP/s on the same card. Short launches pay
// ~7 us of launch, pipeline fill and output besides. Measured against the
// 32 x 64 form (us, operand split and reduction included): Q4_K 9728 -> 2560
// at 777 / 2048 tokens 177 / 361 -> 118 / 245, 2560 -> 19456 at 2048 tokens
// 549 -> 450; the 1.7B Q8_0 prefill of 777 tokens (32-token kernel before)
// 23.1 -> 10.3 ms, the 1.7B Q4_K_M one of 3999 tokens 46.8 -> 42.3 ms.
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
typedef _Float16 H4 __attribute__((ext_vector_type(4)));
typedef _Float16 H8 __attribute__((ext_vector_type(8)));
typedef float F16v __attribute__((ext_vector_type(16)));
typedef uint32_t U2 __attribute__((ext_vector_type(2)));
typedef uint32_t U4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;    // 8 waves
constexpr int kTN = kTiledRows;  // weight rows per workgroup

// 16 bytes at an address that is only 2-byte aligned (Q6_K and Q8_0 blocks
// are 210 and 34 bytes long): one dwordx4 load, which global memory serves at
// any byte alignment.
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

__device__ __forceinline__ uint32_t HalfPair(float v) {
  const _Float16 h = static_cast<_Float16>(v);
  return AsU(H2{h, h});
}

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

// (a & mask) | c with the mask in an SGPR (gfx9 VOP3 takes no literal).
__device__ __forceinline__ uint32_t AndOr(uint32_t a, uint32_t mask, uint32_t c) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(mask), "v"(c));
  return r;
}

// Weight operands of 8 inputs (two dwords of quants), in the operand order
// of SplitX (within every 8 inputs: 0, 2, 1, 3, 4, 6, 5, 7).
//
// Q4_K: q * sc exactly, from the low (mask 0x000F000F) or high (0x00F000F0)
// nibbles. A low nibble read as the f16 1024 + q gives (1024 + q) sc - 1024
// sc; a high nibble in place, 1024 + 16 q, gives (1024 + 16 q) sc/16 - 64 sc;
// the fused multiply-add never rounds (q sc <= 945). sn holds the pair's
// {sc, -1024 sc} or {sc/16, -64 sc} (negated in odd steps).
__device__ __forceinline__ H8 UnpackQ4(uint32_t v0, uint32_t v1, uint32_t mask, uint32_t magic, uint32_t sn) {
  const H2 p = AsH2(sn), sc = H2{p.x, p.x}, nb = H2{p.y, p.y};
  const uint32_t w0 = v0 >> 8, w1 = v1 >> 8;
  const U4 r = {AsU(__builtin_elementwise_fma(AsH2(AndOr(v0, mask, magic)), sc, nb)),
                AsU(__builtin_elementwise_fma(AsH2(AndOr(w0, mask, magic)), sc, nb)),
                AsU(__builtin_elementwise_fma(AsH2(AndOr(v1, mask, magic)), sc, nb)),
                AsU(__builtin_elementwise_fma(AsH2(AndOr(w1, mask, magic)), sc, nb))};
  return __builtin_bit_cast(H8, r);
}
// Q6_K / Q8_0: bytes u read as the f16 1024 + u, less 1024 + kBias: the exact
// u - kBias (q - 32 of Q6_K; q of Q8_0, stored as q + 128), negated if neg.
template <int kBias>
__device__ __forceinline__ H8 UnpackBytes(uint32_t v0, uint32_t v1, uint32_t magic, bool neg) {
  const H2 off = H2{static_cast<_Float16>(1024.0f + kBias), static_cast<_Float16>(1024.0f + kBias)};
  const H2 v[4] = {AsH2(__builtin_amdgcn_perm(magic, v0, 0x04020400u)),
                   AsH2(__builtin_amdgcn_perm(magic, v0, 0x04030401u)),
                   AsH2(__builtin_amdgcn_perm(magic, v1, 0x04020400u)),
                   AsH2(__builtin_amdgcn_perm(magic, v1, 0x04030401u))};
  U4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = AsU(neg ? off - v[i] : v[i] - off);
  return __builtin_bit_cast(H8, r);
}

// QT: the weight type (kQ4_K, kQ6_K or kQ8_0).
//
// A step is 64 inputs of a super-block. For Q4_K, step s holds sub-blocks 2s
// and 2s + 1 (inputs 64 s .. + 64: low and high nibbles of 32 quant bytes).
// For Q6_K, step s = 2 h + m holds strips m and m + 2 of half h (inputs
// 128 h + 32 m + [0, 32) and 128 h + 64 + 32 m + [0, 32): low and high
// nibbles of the same 32 ql bytes, with their qh bits); the token rows are
// staged in that order. For Q8_0, two 32-weight blocks.
//
// kTM: tokens per workgroup. 128: waves in 2 token halves x 4 row quarters,
// each 64 tokens x 64 rows; 64 (segments of up to 64 tokens, half the
// products of a 128-token tile): 8 row eighths, each 64 tokens x 32 rows.
template <int QT, int kTM>
struct TileLds {
  static constexpr bool kQ4 = QT == kQ4_K, kQ6 = QT == kQ6_K;
  // quants of a step, 16-byte chunks side by side over the rows (a wave's
  // reads of one chunk are 512 consecutive bytes):
  //  Q4_K [stage][h][row]: bytes 16 h .. + 16 of the row's 32;
  //  else [stage][2 p + h][row]: unsigned bytes, inputs 8 h .. + 8 of slices
  //  2 p and 2 p + 1 (slice: 16 inputs of the step)
  U4 Bq[2][kQ4 ? 2 : 4][kTN];
  // Q4_K [table][step][row]: UnpackQ4's pairs of the step's two sub-blocks
  U2 S4[kQ4 ? 2 : 1][4][kQ4 ? kTN : 1];
  _Float16 Ss[kQ4 ? 2 : 1][2][kQ4 ? kTM : 1][8];  // Q4_K [table][hi, lo][token]: sub-block sums
  _Float16 Mn[kQ4 ? 2 : 1][kQ4 ? kTN : 1][8];     // Q4_K [table][row]: integer mins
  float2 Dd[kQ4 ? 2 : 1][kQ4 ? kTN : 1];          // Q4_K [table][row]: d, -32 dmin
  // Q6_K [4 table + step][row]: d * sc of the step's 4 slices; Q8_0
  // [stage][row]: d of its 2 blocks
  static constexpr int kSc = kQ4 ? 1 : kQ6 ? 4 : 2;
  alignas(16) float Sc[kQ4 ? 1 : kQ6 ? 8 : 2][kQ4 ? 1 : kTN][kSc];
  alignas(16) float Is[kTM];  // 1 / s of the token rows
};

// Part zt of the tile's K (zt < 0: this launch's part blockIdx.y), tile (tm,
// nt) of job j. As0, As1: a stage's token rows [hi, lo][token] each, swizzled
// (ASwz): one array per stage, since the compiler tells LDS arrays apart when
// it places the waits for its DMA loads, so that reads of one stage do not
// wait for the DMA into the other.
template <int QT, int kTM>
__device__ __forceinline__ void TGemmTile(const TiledArgs& a, int wgi, int zt, int tm, int nt, int j,
                                          _Float16 (&As0)[2][kTM][64], _Float16 (&As1)[2][kTM][64],
                                          TileLds<QT, kTM>& L) {
  constexpr bool kQ4 = QT == kQ4_K, kQ6 = QT == kQ6_K;
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

  // Two stages (a step's operands) alternate; the per-super-block tables of
  // Q4_K and Q6_K alternate with the super-block.
  auto as = [&](int st) -> _Float16(*)[kTM][64] { return st ? As1 : As0; };
  auto& Bq = L.Bq;
  auto& S4 = L.S4;
  auto& Ss = L.Ss;
  auto& Mn = L.Mn;
  auto& Dd = L.Dd;
  auto& Sc = L.Sc;
  auto& Is = L.Is;

  // The weight row this thread stages, as local row br, and the half bq of a
  // step (Q4_K: 16 of its 32 quant bytes; Q6_K: ql / qh bytes 16 bq .. + 16,
  // slices bq and 2 + bq; Q8_0: block bq, slices 2 bq and 2 bq + 1). A pair's
  // workgroup holds 128 output rows; even waves stage gate rows, odd ones up
  // rows (the matrix is wave-uniform). A wave's rows are gate rows and then
  // the same up rows: 32 + 32 as its two tiles, or 16 + 16 of its one.
  const int bq = tid & 1, bi = (tid >> 1) & 31;
  const int pr = 32 * (wave >> 1) + bi;  // (pair: row of the 128)
  const int br = kNI == 1 && pair ? 32 * (pr >> 4) + 16 * (wave & 1) + (pr & 15) : tid >> 1;
  const uint8_t* bmat = (pair && (wave & 1)) ? a.job[1].w.w : J.w.w;
  const int brow_i = pair ? min(128 * nt + pr, rows - 1) : min(kTN * nt + br, rows - 1);
  const Rsrc rwt = MakeRsrc(bmat, static_cast<uint32_t>(rows) * static_cast<uint32_t>(rb));
  const uint32_t b_off = static_cast<uint32_t>(brow_i) * static_cast<uint32_t>(rb);
  // (Q6_K, Q8_0: 2-byte aligned global loads, a uniform base and a 32-bit
  // lane offset)
  const uint32_t b_lane = b_off + (kQ6 ? 16u : 34u) * bq;
  // The token rows of a step reach LDS by DMA (buffer loads with an LDS
  // destination: a wave's 64 lanes x 16 bytes land as 1 KB in a row). A
  // step's rows are 2 parts x kTM tokens x 128 bytes = kTM / 4 such loads,
  // kDma per wave: load i of wave w fills part w / 4, rows 8 b .. 8 b + 7, b =
  // (kDma w + i) % (kTM / 8); lane L reads token row 8 b + L / 8 and lands at chunk
  // L % 8 of it, which holds logical chunk (L % 8) ^ ASwz(row). Logical chunk
  // c holds step inputs 8 c .. + 8 (Q6_K: 8 c and 32 + 8 c of the step's two
  // strips). The buffer resources end at the last token, so the rows past it
  // read as zeros.
  const uint32_t a_bytes = static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 2u;
  const Rsrc ra_src = MakeRsrc(wave < 4 ? x.hi : x.lo, a_bytes);
  uint32_t a_voff[kDma];
#pragma unroll
  for (int i = 0; i < kDma; ++i) {
    const int r = 8 * ((kDma * wave + i) & (kTM / 8 - 1)) + (lane >> 3);
    const int lc = (lane & 7) ^ ASwz(r);
    a_voff[i] = (static_cast<uint32_t>(m0 + r) * static_cast<uint32_t>(K) + 8u * lc + (kQ6 && lc >= 4 ? 32u : 0u)) * 2u;
  }
  // Q4_K sub-block sums: part x token, one chunk of 8 (threads 2 kTM ..
  // repeat the first)
  const int sp = (wave / kNI) & 1, sr = tid & (kTM - 1);
  const Rsrc rsum = MakeRsrc(sp ? x.sum_lo : x.sum_hi, static_cast<uint32_t>(M) * static_cast<uint32_t>(K >> 5) * 2u);
  const uint32_t s_off = static_cast<uint32_t>(m0 + sr) * static_cast<uint32_t>(K >> 5) * 2u;

  uint32_t mlo, mhi, magic;
  asm volatile("s_mov_b32 %0, 0xf000f" : "=s"(mlo));
  asm volatile("s_mov_b32 %0, 0xf000f0" : "=s"(mhi));
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
  const uint32_t magic8 = 0x64646464u;

  // The weights' loads run kAhead steps ahead in a register ring (three; two
  // for Q6_K, which has no registers for a second slot): step g's quant bytes
  // sit in slot g % kSlots from their issue until they are staged; a
  // super-block's first step also loads its header (Q4_K: d, dmin, scales;
  // Q6_K: scales, d) and the tokens' sub-block sums. Every step issues the
  // same loads, unconditionally (steps past the end re-read the last one), so
  // the compiler counts them and waits for one step's loads while the next
  // steps' stay in flight.
  U4 hn = {}, sn = {};
  constexpr int kAhead = kQ6 ? 2 : 3, kSlots = kAhead - 1;
  U4 rl[kSlots], rh[kSlots];  // quant bytes (Q4_K: rl alone)
  uint32_t rd[kSlots];        // Q8_0 d
  uint32_t dn = 0;            // Q6_K d
  const int nsteps = 4 * (o1 - o0);
  // VMEM instructions of one issue() of a super-block's first step (ss == 0)
  // and of the others (the counts of the compiled code; fewer would only wait
  // longer, more would let a step read rows still in flight)
  constexpr int kLoads0 = kQ4 ? 3 : kQ6 ? 4 : 3, kLoads1 = kQ4 ? 1 : kQ6 ? 2 : 3;
  // the token rows of step g (g = 4 o + s of this part, super-block o0 + o)
  // into stage st
  auto issue_a = [&](int g, int st) {
    g = min(g, nsteps - 1);
    const int ob = o0 + (g >> 2), s = g & 3;
    const int so = kQ6 ? 2 * (256 * ob + 128 * (s >> 1) + 32 * (s & 1)) : 2 * (256 * ob + 64 * s);
#pragma unroll
    for (int i = 0; i < kDma; ++i)
      DmaLds(ra_src, &as(st)[wave >> 2][8 * ((kDma * wave + i) & (kTM / 8 - 1))][0], a_voff[i], so);
  };
  // (ss = g % 4, known at compile time at every call)
  auto issue = [&](int g, int slot, int ss) {
    g = min(g, nsteps - 1);
    const int ob = o0 + (g >> 2), s = g & 3;
    if constexpr (kQ4) {
      rl[slot] =
          __builtin_bit_cast(U4, __builtin_amdgcn_raw_buffer_load_b128(rwt, b_off + 16 + 16 * bq, 144 * ob + 32 * s, 0));
      if (ss == 0) {
        hn = __builtin_bit_cast(U4, __builtin_amdgcn_raw_buffer_load_b128(rwt, b_off, 144 * ob, 0));
        sn = __builtin_bit_cast(U4, __builtin_amdgcn_raw_buffer_load_b128(rsum, s_off, 16 * ob, 0));
      }
    } else if constexpr (kQ6) {
      const uint8_t* blk = bmat + 210 * static_cast<int64_t>(ob);
      rl[slot] = GLoad<U4A2>(blk + 64 * (s >> 1) + 32 * (s & 1) + b_lane);
      rh[slot] = GLoad<U4A2>(blk + 128 + 32 * (s >> 1) + b_lane);
      if (ss == 0) {
        hn = GLoad<U4A2>(blk + 192 + b_off);
        dn = GLoad<uint16_t>(blk + 208 + b_off);
      }
    } else {
      const uint8_t* blk = bmat + 34 * static_cast<int64_t>(8 * ob + 2 * s);
      rl[slot] = GLoad<U4A2>(blk + 2 + b_lane);
      rh[slot] = GLoad<U4A2>(blk + 18 + b_lane);
      rd[slot] = GLoad<uint16_t>(blk + b_lane);
    }
  };
  // the tables of a super-block (table tb), from its header and sums; the
  // row's two threads take sub-blocks 4 bq .. + 4
  auto store_tables = [&](int tb) {
    if constexpr (kQ4) {
      // (unconditional stores, some of one value by two threads)
      *reinterpret_cast<U4*>(&Ss[tb][sp][sr][0]) = sn;
      const uint32_t b0 = hn.y, b4 = hn.z, b8 = hn.w;
      const uint32_t sc4 = bq ? (b8 & 0x0F0F0F0Fu) | ((b0 >> 2) & 0x30303030u) : b0 & 0x3F3F3F3Fu;
      const uint32_t mn4 = bq ? ((b8 >> 4) & 0x0F0F0F0Fu) | ((b4 >> 2) & 0x30303030u) : b4 & 0x3F3F3F3Fu;
      // signs: step 2 bq + i, super-block
      const uint32_t neg_sb = tb ? 0x80008000u : 0u;
      U2 m;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float f0 = static_cast<float>((sc4 >> (16 * i)) & 0xFFu);
        float f1 = static_cast<float>((sc4 >> (16 * i + 8)) & 0xFFu);
        if (i == 1) f0 = -f0, f1 = -f1;
        S4[tb][2 * bq + i][br] =
            U2{AsU(H2{static_cast<_Float16>(f0), static_cast<_Float16>(-1024.0f * f0)}),
               AsU(H2{static_cast<_Float16>(0.0625f * f1), static_cast<_Float16>(-64.0f * f1)})};
        m[i] = AsU(H2{static_cast<_Float16>(static_cast<float>((mn4 >> (16 * i)) & 0xFFu)),
                      static_cast<_Float16>(static_cast<float>((mn4 >> (16 * i + 8)) & 0xFFu))}) ^ neg_sb;
      }
      *reinterpret_cast<U2*>(&Mn[tb][br][4 * bq]) = m;
      Dd[tb][br] = float2{dev::HalfToFloatFast(hn.x & 0xFFFFu),
                          (tb ? 32.0f : -32.0f) * dev::HalfToFloatFast(hn.x >> 16)};
    } else if constexpr (kQ6) {
      // slices bq and 2 + bq of each step: scale sc[8 h + 2 k + l / 16] of
      // strip k = m + 2 p, l = 16 bq
      const float d = dev::HalfToFloatFast(dn);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int si = 8 * (s >> 1) + 2 * ((s & 1) + 2 * p);
          const uint32_t w = hn[si >> 2] >> (8 * (si & 3));
          Sc[4 * tb + s][br][2 * p + bq] =
              d * static_cast<float>(static_cast<int8_t>((bq ? w >> 8 : w) & 0xFFu));
        }
    }
  };
  // the quants of a step (sub-step s of its super-block) into stage st
  auto store_b = [&](int slot, int s, int st) {
    if constexpr (kQ4) {
      Bq[st][bq][br] = rl[slot];
    } else if constexpr (kQ6) {
      // ql bytes: low nibbles strip 0 (slice bq), high nibbles strip 1 (slice
      // 2 + bq); their qh bits at 2 m and 2 m + 4
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int k = (s & 1) + 2 * p;
        U4 q;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          q[i] = ((rl[slot][i] >> (4 * p)) & 0x0F0F0F0Fu) | (((rh[slot][i] >> (2 * k)) & 0x03030303u) << 4);
        reinterpret_cast<U2*>(&Bq[st][2 * p][br])[bq] = U2{q.x, q.y};
        reinterpret_cast<U2*>(&Bq[st][2 * p + 1][br])[bq] = U2{q.z, q.w};
      }
    } else {
      const uint32_t f = 0x80808080u;
      const U4 q0 = rl[slot], q1 = rh[slot];
      Bq[st][2 * bq][br] = U4{q0.x ^ f, q0.y ^ f, q1.x ^ f, q1.y ^ f};
      Bq[st][2 * bq + 1][br] = U4{q0.z ^ f, q0.w ^ f, q1.z ^ f, q1.w ^ f};
      Sc[st][br][bq] = dev::HalfToFloatFast(rd[slot]);
    }
  };

  // A scale group (Q4_K: a step; Q8_0: a block; Q6_K: a slice, its sub-block)
  // accumulates in P from zero and is scaled into T while the next group's
  // products run (the first time it adds zeros). kGroup slices multiply the
  // tokens' lo parts, then the hi parts: lo products added to sums of the hi
  // parts' size round at that size, which over long chains measured two to
  // three times the error.
  // The matrix core rounds its sums down (measured: a common negative error
  // of every token, which an attention average keeps where it averages the
  // tokens' own errors out), so every odd group multiplies the negated
  // weights and is subtracted: the two halves' errors cancel. The min terms
  // alternate by super-block.
  constexpr int kGl = kQ6 ? 0 : 1, kGroup = 1 << kGl;
  F16v T[2][kNI], P[2][kNI];
  float Cs[kNI] = {};
#pragma unroll
  for (int i = 0; i < 2 * kNI; ++i) {
    T[i / kNI][i % kNI] = F16v{};
    P[i / kNI][i % kNI] = F16v{};
  }

  // token operands of one slice and part, double-buffered; the weight
  // operands of a group
  H8 op[2][2], b[kGroup][kNI];
  // quants of the wave's rows (and Q4_K scale pairs, Q6_K / Q8_0 scales):
  // Q4_K a whole step; else slices 2 p and 2 p + 1
  U4 qv[kNI];
  U2 s4[kNI];
  float sc[kNI][2];
  // Q4_K's lane half lh takes quant bytes 16 lh .. + 16: slice kk multiplies
  // logical token chunk 4 (kk / 2) + 2 lh + kk % 2, else 2 kk + lh
  auto read_a = [&](H8* q, int st, int part, int kk) {
    const int lc = kQ4 ? 4 * (kk >> 1) + 2 * lh + (kk & 1) : 2 * kk + lh;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
      const int ar = 64 * wm + 32 * mi + l32;
      q[mi] = *reinterpret_cast<const H8*>(&as(st)[part][ar][8 * (lc ^ ASwz(ar))]);
    }
  };
  auto read_q = [&](int st, int p, int tb, int s) {
#pragma unroll
    for (int ni = 0; ni < kNI; ++ni) {
      const int r = kWN * wn + 32 * ni + l32;
      qv[ni] = Bq[st][kQ4 ? lh : 2 * p + lh][r];
      if constexpr (kQ4) {
        s4[ni] = S4[tb][s][r];
      } else if constexpr (kQ6) {
        const float2 v = *reinterpret_cast<const float2*>(&Sc[4 * tb + s][r][2 * p]);
        sc[ni][0] = v.x, sc[ni][1] = v.y;
      } else {
        sc[ni][0] = Sc[st][r][p];
      }
    }
  };

  // (read again by the epilogue from LDS: loads there would wait for its
  // stores)
  if (tid < kTM) Is[tid] = x.inv_s[min(m0 + tid, M - 1)];
  // prologue: step 0 staged, step 1's token rows and weights and step 2's
  // weights in flight
  issue_a(0, 0);
  issue(0, 0, 0);
  if constexpr (kAhead == 3) issue(1, 1, 1);
  store_tables(0);
  store_b(0, 0, 0);
  issue(kAhead - 1, 0, kAhead - 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  issue_a(1, 1);
  read_a(op[0], 0, 1, 0);
  read_q(0, 0, 0, 0);
  if constexpr (kQ4) {
#pragma unroll
    for (int ni = 0; ni < kNI; ++ni) sc[ni][0] = Dd[0][kWN * wn + 32 * ni + l32].x;
  }
  for (int o = 0; o < o1 - o0; ++o) {
    const int tb = o & 1;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      // step g = 4 o + s multiplies stage s % 2 while step g + 1's weights are
      // staged into the other one, where its token rows' DMA, issued a step
      // ago, lands. The barrier sits before the last of the step's 8 items (a
      // slice and part), whose operands are in registers by then: past it the
      // next step's first operands are read while that item multiplies, and
      // step g + 2's DMA is issued.
      const int g = 4 * o + s, st = s & 1, nx = st ^ 1, ns = (s + 1) & 3;
      // Q4_K, the super-block's end: its mins, -32 dmin and sub-block sums
      H8 bm[kNI], xs[2];
      float dm[kNI];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int kk = ((i >> (kGl + 1)) << kGl) | (i & (kGroup - 1)), hi = (i >> kGl) & 1;
        const int kg = kk & (kGroup - 1);
        if (i == 7) {
          // step g + 1's token rows have landed (only the weight loads issued
          // in this step, after them, may still be in flight)
          if (s == (4 - kAhead))
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads0) : "memory");
          else
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads1) : "memory");
          __syncthreads();
          if (kQ4 && s == 3) {
#pragma unroll
            for (int t = 0; t < kNI; ++t) {
              const int r = kWN * wn + 32 * t + l32;
              bm[t] = *reinterpret_cast<const H8*>(&Mn[tb][r][0]);
              dm[t] = Dd[tb][r].y;  // (its sign the mins')
              sc[t][0] = Dd[tb ^ 1][r].x;
            }
#pragma unroll
            for (int mi = 0; mi < 2; ++mi)
              xs[mi] = *reinterpret_cast<const H8*>(&Ss[tb][lh][64 * wm + 32 * mi + l32][0]);
          }
          read_a(op[0], nx, 1, 0);
        } else {
          const int k1 = (((i + 1) >> (kGl + 1)) << kGl) | ((i + 1) & (kGroup - 1)), h1 = ((i + 1) >> kGl) & 1;
          read_a(op[(i + 1) & 1], st, h1 ^ 1, k1);
        }
        if (!hi) {
#pragma unroll
          for (int ni = 0; ni < kNI; ++ni) {
            const uint32_t v0 = qv[ni][2 * (kk & 1)], v1 = qv[ni][2 * (kk & 1) + 1];
            if constexpr (kQ4)
              b[kg][ni] = UnpackQ4(v0, v1, kk < 2 ? mlo : mhi, magic, kk < 2 ? s4[ni].x : s4[ni].y);
            else
              b[kg][ni] = UnpackBytes<kQ6 ? 32 : 128>(v0, v1, magic8, (kk >> kGl) & 1);
          }
        }
        const H8* q = op[i & 1];
        const bool fresh = !hi && kg == 0 && !(kQ4 && kk > 0);
        const bool last_neg = kQ4 ? (s & 1) == 0 : ((kk >> kGl) & 1) == 0;  // P's group was an odd one
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
          for (int ni = 0; ni < kNI; ++ni) Cs[ni] = sc[ni][kQ6 ? kk & 1 : 0];
        }
        // the next step's staging, spread over the items
        if (i == 1 && s == 3) store_tables(tb ^ 1);  // step g + 1 starts super-block o + 1
        if (i == 3 && !kQ4) read_q(st, 1, tb, s);
        if (i == 3) store_b(ns % kSlots, ns, nx);
        if (i == 4) issue(g + kAhead, ns % kSlots, (s + kAhead) & 3);
        if (i == 7) {
          read_q(nx, 0, s == 3 ? tb ^ 1 : tb, ns);
          // (the DMA after these reads, which the compiler would else make
          // wait for it)
          __builtin_amdgcn_sched_barrier(0);
          issue_a(g + 2, st);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (kQ4 && s == 3) {
        // the min term: T -= 32 dmin * sum_j m_j * S_j, the 8 hi sums in the
        // lower lane half's k, the 8 lo sums in the upper's
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
          for (int ni = 0; ni < kNI; ++ni) {
            const F16v qm = MmaFresh(xs[mi], bm[ni]);
#pragma unroll
            for (int v = 0; v < 16; ++v) T[mi][ni][v] = __builtin_fmaf(dm[ni], qm[v], T[mi][ni][v]);
          }
        }
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

// A launch over jobs of type QA, or of QA and QB (Q4_K and Q6_K: a layer's q, k
// and v in one launch; as two launches on two streams they cost ~20 us of
// cross-stream waits per layer).
template <int QA, int QB, int kTM>
__global__ __launch_bounds__(kThreads) void TGemmKernel(TiledArgs a) {
  using LA = TileLds<QA, kTM>;
  using LB = TileLds<QB, kTM>;
  __shared__ __align__(16) _Float16 As0[2][kTM][64];
  __shared__ __align__(16) _Float16 As1[2][kTM][64];
  __shared__ __align__(16) uint8_t rest[sizeof(LA) > sizeof(LB) ? sizeof(LA) : sizeof(LB)];
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
  if (QA == QB || a.job[j].w.type == QA)
    TGemmTile<QA, kTM>(a, wgi, zt, tm, nt, j, As0, As1, *reinterpret_cast<LA*>(rest));
  else
    TGemmTile<QB, kTM>(a, wgi, zt, tm, nt, j, As0, As1, *reinterpret_cast<LB*>(rest));
}

// The tail tiles of a pair launch: y = silu(g) * u with g, u the sums of the
// tile's K parts (added in part order, then scaled as the full tiles' sums
// are), the full tiles' SwiGLU arithmetic. Workgroup (tile, y) takes tokens
// 8 y .. 8 y + 7 of the tile, four outputs per thread.
constexpr int kTailPer = 4;
template <int kTM>
__global__ __launch_bounds__(256) void TailSwiGLUKernel(TiledArgs a) {
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
    // (tokens past M were not stored: their sums are read but not used)
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

void LaunchTiled(const TiledArgs& a, hipStream_t s) {
  int tiles = 0;
  for (int j = 0; j < a.n_jobs; ++j) tiles += a.tiles[j];
  const uint32_t type = a.job[0].w.type;
  RPG_CHECK(type == kQ4_K || type == kQ6_K || type == kQ8_0, "tiled gemm: weight type %u", type);
  bool mixed = false;
  for (int j = 1; j < a.n_jobs + (a.pair ? 1 : 0); ++j) {
    const uint32_t tj = a.job[j].w.type;
    RPG_CHECK(tj == type || (!a.pair && TiledMixes(tj) && TiledMixes(type)), "tiled gemm: types %u and %u in one launch",
              type, tj);
    mixed = mixed || tj != type;
  }
  RPG_CHECK(a.x.K % 256 == 0 && a.x.K >= 256, "tiled gemm: K = %d is not a multiple of 256", a.x.K);
  RPG_CHECK(a.tokens == TiledTokens(a.x.M) && a.tiles_m == CeilDiv(a.x.M, a.tokens), "tiled gemm: bad token tiles");
  RPG_CHECK(a.ksplit >= 1 && a.ksplit <= a.x.K / 256, "tiled gemm: bad K split %d", a.ksplit);
  const int total = tiles * a.tiles_m;
  const int n_tail = a.tail_split > 1 ? total - a.tail_wg : 0;
  if (a.tail_split > 1)
    RPG_CHECK(a.pair && a.ksplit == 1 && a.tail_wg >= 0 && a.tail_wg < total && a.tail_split <= a.x.K / 256 &&
                  static_cast<int64_t>(n_tail) * a.tail_split * a.tokens * kTN <= a.x.part_floats,
              "tiled gemm: bad tail split %d from workgroup %d of %d", a.tail_split, a.tail_wg, total);
  const dim3 grid(static_cast<unsigned>(total + n_tail * (a.tail_split - 1)), static_cast<unsigned>(a.ksplit));
  const bool small = a.tokens == 64;
  const dim3 block(kThreads);
  if (mixed) {
    if (small)
      hipLaunchKernelGGL((TGemmKernel<kQ4_K, kQ6_K, 64>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((TGemmKernel<kQ4_K, kQ6_K, 128>), grid, block, 0, s, a);
  } else if (type == kQ4_K) {
    if (small)
      hipLaunchKernelGGL((TGemmKernel<kQ4_K, kQ4_K, 64>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((TGemmKernel<kQ4_K, kQ4_K, 128>), grid, block, 0, s, a);
  } else if (type == kQ6_K) {
    if (small)
      hipLaunchKernelGGL((TGemmKernel<kQ6_K, kQ6_K, 64>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((TGemmKernel<kQ6_K, kQ6_K, 128>), grid, block, 0, s, a);
  } else {
    if (small)
      hipLaunchKernelGGL((TGemmKernel<kQ8_0, kQ8_0, 64>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((TGemmKernel<kQ8_0, kQ8_0, 128>), grid, block, 0, s, a);
  }
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
