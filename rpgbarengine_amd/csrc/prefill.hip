// Prefill projections on the gfx950 matrix cores (v_mfma_f32_16x16x32_f16);
// the operand construction that keeps them exact is described in prefill.h.
//
// The tiled GEMM (gemm_tiled.hip) takes every matrix whose width is a
// multiple of 256. QGemm8Kernel here serves the other Q8_0 widths: 2 waves
// over 64 tokens x 128 rows, the token operands of a 64-input step (both f16
// parts) staged in LDS once for the workgroup, every lane assembling its
// weight operand from the raw quant bytes, the next step's loads in flight
// while the current one is multiplied.
//
// MFMA operand layout (16x16x32 f16): lane l holds A[i = l % 16][8*(l/16) ..
// +8), B[8*(l/16) .. +8][j = l % 16]; the result C[4*(l/16) + e][l % 16],
// e < 4.

#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "common.h"
#include "lanes.h"
#include "expf_glibc.h"
#include "prefill.h"
#include "quant_dev.h"

namespace rpg {
namespace k {

namespace {

typedef _Float16 H2 __attribute__((ext_vector_type(2)));
typedef _Float16 H4 __attribute__((ext_vector_type(4)));
typedef _Float16 H8 __attribute__((ext_vector_type(8)));
typedef float F4 __attribute__((ext_vector_type(4)));
typedef uint32_t U2 __attribute__((ext_vector_type(2)));
typedef uint32_t U4 __attribute__((ext_vector_type(4)));
// 8 bytes at an address that is only 2-byte aligned (Q6_K and Q8_0 blocks
// are 210 and 34 bytes long): one dwordx2 load, which global memory serves
// at any byte alignment.
typedef U2 U2A2 __attribute__((aligned(2)));

template <typename T>
__device__ __forceinline__ T GLoad(const void* p) {
  return *(const __attribute__((address_space(1))) T*)(p);
}

__device__ __forceinline__ H2 AsH2(uint32_t v) { return __builtin_bit_cast(H2, v); }
__device__ __forceinline__ uint32_t AsU(H2 v) { return __builtin_bit_cast(uint32_t, v); }

// ---------------------------------------------------------------- SplitRows

constexpr int kSplitThreads = 256;      // rows of up to 10240 inputs
constexpr int kSplitThreadsWide = 1024;  // wider rows, up to 40960 inputs
constexpr int kSplitChunks = 5;          // 8-input chunks per thread at most
constexpr int kSplitPendMax = 8;         // pending split-K partials a row may carry

template <int NW>
__device__ __forceinline__ float BlockMax(float v, float* red) {
  v = lanes::WaveMaxF(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float m = red[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) m = fmaxf(m, red[i]);
  return m;
}
// the waves' partial sums added pairwise: ((r0 + r1) + (r2 + r3)) for four
template <int NW>
__device__ __forceinline__ double PairSum(const double* r) {
  if constexpr (NW == 1)
    return r[0];
  else
    return PairSum<NW / 2>(r) + PairSum<NW / 2>(r + NW / 2);
}

// One workgroup of NT threads per token row; NC 8-input chunks per thread
// (K <= 8 NT NC). kNorm: RMSNorm with gain norm_w; kPend > 0: up to kPend
// pending split-K partials are added first. The prologue's loads (inputs, gains,
// partials) carry no branches, so all of them are in flight before the
// first is used.
template <int NT, int NC, bool kNorm, int kPend>
__global__ __launch_bounds__(NT) void SplitRowsKernel(float* X, int64_t ldx, int K, const float* __restrict__ norm_w,
                                                      float eps, SplitX o, SplitPending pend) {
  constexpr int NW = NT / 64;
  const int t = blockIdx.x, tid = threadIdx.x;
  const float4* x4 = reinterpret_cast<const float4*>(X + t * ldx);
  const int n8 = K >> 3;
  __shared__ double redd[NW];
  __shared__ float redf[NW];
  float v[NC][8];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int ch = min(tid + c * NT, n8 - 1);
    const float4 a = x4[2 * ch], b = x4[2 * ch + 1];
    v[c][0] = a.x, v[c][1] = a.y, v[c][2] = a.z, v[c][3] = a.w;
    v[c][4] = b.x, v[c][5] = b.y, v[c][6] = b.z, v[c][7] = b.w;
  }
  // the RMSNorm gain chunks load with the inputs (used after the sum of
  // squares)
  float wv[NC][8];
  if constexpr (kNorm) {
    const float4* w4 = reinterpret_cast<const float4*>(norm_w);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int ch = min(tid + c * NT, n8 - 1);
      const float4 a = w4[2 * ch], b = w4[2 * ch + 1];
      wv[c][0] = a.x, wv[c][1] = a.y, wv[c][2] = a.z, wv[c][3] = a.w;
      wv[c][4] = b.x, wv[c][5] = b.y, wv[c][6] = b.z, wv[c][7] = b.w;
    }
  }
  if constexpr (kPend > 0) {
    // x += the sum of the split partials in split order (SplitKReduceKernel's
    // arithmetic), written back as the residual. Every partial of a chunk
    // (of every chunk, up to two per thread) is requested before any is
    // added: one round trip, not one per split. Split z >= ksplit reloads the
    // last one (an address in bounds) and is not added.
    constexpr int kGroup = NC * kPend <= 8 ? NC : 1;  // chunks whose partials are in flight together
    const int nz = pend.ksplit;
#pragma unroll
    for (int c0 = 0; c0 < NC; c0 += kGroup) {
      float4 pp[kGroup][kPend][2];
#pragma unroll
      for (int g = 0; g < kGroup; ++g) {
        const int ch = min(tid + (c0 + g) * NT, n8 - 1);
#pragma unroll
        for (int z = 0; z < kPend; ++z) {
          const int zz = min(z, nz - 1);
          const float4* p4 = reinterpret_cast<const float4*>(
              pend.part + (static_cast<int64_t>(zz) * pend.M + t) * pend.part_ld + pend.pcol + 8 * ch);
          pp[g][z][0] = p4[0];
          pp[g][z][1] = p4[1];
        }
      }
#pragma unroll
      for (int g = 0; g < kGroup; ++g) {
        const int c = c0 + g, ch = tid + c * NT;
        float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int z = 0; z < kPend; ++z) {
          if (z == 0 || z < nz) {  // nz >= 1
            const float4 a = pp[g][z][0], b = pp[g][z][1];
            sum[0] += a.x, sum[1] += a.y, sum[2] += a.z, sum[3] += a.w;
            sum[4] += b.x, sum[5] += b.y, sum[6] += b.z, sum[7] += b.w;
          }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) v[c][i] = v[c][i] + sum[i];
        if (ch < n8) {
          float4* xo = reinterpret_cast<float4*>(X + t * ldx) + 2 * ch;
          xo[0] = make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
          xo[1] = make_float4(v[c][4], v[c][5], v[c][6], v[c][7]);
        }
      }
    }
  }
  if constexpr (kNorm) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (tid + c * NT < n8)
#pragma unroll
        for (int i = 0; i < 8; ++i) s += static_cast<double>(v[c][i]) * v[c][i];
    s = lanes::WaveSumD(s);
    if ((tid & 63) == 0) redd[tid >> 6] = s;
    __syncthreads();
    const double total = PairSum<NW>(redd);
    const float scale =
        static_cast<float>(1.0 / __builtin_sqrt(total / static_cast<double>(K) + static_cast<double>(eps)));
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) v[c][i] = __fmul_rn(__fmul_rn(v[c][i], scale), wv[c][i]);
  }
  float mx = 0.0f;
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (tid + c * NT < n8)
#pragma unroll
      for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(v[c][i]));
  mx = BlockMax<NW>(mx, redf);
  // s = 2^(15 - E) for max = f * 2^E, f in [0.5, 1): max * s in [2^14, 2^15)
  int e = 0;
  (void)frexpf(mx, &e);
  const int se = mx > 0.0f ? min(max(15 - e, -100), 100) : 0;
  const float s = ldexpf(1.0f, se), s32 = ldexpf(1.0f, se - 5);
  if (tid == 0) o.inv_s[t] = ldexpf(1.0f, -se);
  _Float16* hi = static_cast<_Float16*>(o.hi) + static_cast<int64_t>(t) * K;
  _Float16* lo = static_cast<_Float16*>(o.lo) + static_cast<int64_t>(t) * K;
  _Float16* shi = static_cast<_Float16*>(o.sum_hi) + static_cast<int64_t>(t) * (K >> 5);
  _Float16* slo = static_cast<_Float16*>(o.sum_lo) + static_cast<int64_t>(t) * (K >> 5);
  constexpr int kPerm[8] = {0, 2, 1, 3, 4, 6, 5, 7};
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int ch = tid + c * NT;
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) sum += v[c][i];
    // sum of the 32 inputs of this chunk's sub-block: chunks 4j..4j+3 sit
    // on 4 consecutive lanes
    sum += lanes::DppF<lanes::kQuadXor1>(sum);
    sum += lanes::DppF<lanes::kQuadXor2>(sum);
    if (ch < n8) {
      H8 h, l;
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        const float xs = v[c][kPerm[p]] * s;
        const _Float16 xh = static_cast<_Float16>(xs);
        h[p] = xh;
        l[p] = static_cast<_Float16>(xs - static_cast<float>(xh));
      }
      *reinterpret_cast<H8*>(hi + 8 * ch) = h;
      *reinterpret_cast<H8*>(lo + 8 * ch) = l;
      if ((ch & 3) == 0) {
        const float ss = sum * s32;
        const _Float16 sh = static_cast<_Float16>(ss);
        shi[ch >> 2] = sh;
        slo[ch >> 2] = static_cast<_Float16>(ss - static_cast<float>(sh));
      }
    }
  }
}

// ---------------------------------------------------------------- QGemm

constexpr int kGT = 128;             // threads per workgroup (2 waves)
constexpr int kTM = 64;              // tokens per workgroup
constexpr int kWN = 64;              // weight rows per wave
constexpr int kTN = 2 * kWN;         // weight rows per workgroup
constexpr int kStep = 64;            // inputs per pipeline step
constexpr int kARow = kStep + 8;     // LDS row of one token's step (f16, padded)

constexpr int kGemmSplitMax = 4;     // K splits of one product (partials summed in order)
constexpr int kTiledSplitMax = kMaxPendParts;  // those of a tiled launch
static_assert(kGemmSplitMax <= kTiledSplitMax && kTiledSplitMax <= kSplitPendMax, "SplitRows holds every pending partial of a chunk in flight");

struct GemmArgs {
  SplitX x;
  GemmJob job[3];
  int32_t tiles[3];  // N tiles per job
  int32_t n_jobs;
  int32_t ksplit;    // blockIdx.z takes super-blocks [z * n / ksplit, (z + 1) * n / ksplit)
  int64_t part_ld;   // partials: x.part[(z * M + token) * part_ld + pcol[job] + row]
  int32_t pcol[3];
};

// The SplitX of the super-blocks [o0, ...): the same rows, pointers moved.
__device__ __forceinline__ SplitX ShiftSplit(const SplitX& x, int k0) {
  SplitX r = x;
  r.hi = static_cast<_Float16*>(x.hi) + k0;
  r.lo = static_cast<_Float16*>(x.lo) + k0;
  r.sum_hi = static_cast<_Float16*>(x.sum_hi) + (k0 >> 5);
  r.sum_lo = static_cast<_Float16*>(x.sum_lo) + (k0 >> 5);
  return r;
}

// Result of one output element: to y (with the job's epilogue), or to the
// split-K partials.
__device__ __forceinline__ void PutOut(const GemmJob& J, const SplitX& x, float* part, int64_t part_ld, int pcol,
                                       int ksplit, int z, int tok, int row, float v) {
  if (ksplit > 1) {
    part[(static_cast<int64_t>(z) * x.M + tok) * part_ld + pcol + row] = v;
  } else {
    float* y = J.y + static_cast<int64_t>(tok) * J.ldy + row;
    *y = J.epi == kAdd ? *y + v : v;
  }
}

// Staged token operands of one step: [part][token][2 segments of 32 inputs]
// f16, 16-byte chunks: 2 parts x 64 tokens x 8 chunks = 1024 chunks, 8 per
// thread. Segment s starts at input k[s] (the two 32-input K-steps of a step
// need not be adjacent).
struct AStage {
  U4 c[8];
};

__device__ __forceinline__ void LoadA(AStage& st, const SplitX& x, int m0, int k0, int k1) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int idx = tid + i * kGT;              // 0..1023
    const int part = idx >> 9, r = (idx >> 3) & 63, ch = idx & 7;
    const int tok = min(m0 + r, x.M - 1);
    const _Float16* src = static_cast<const _Float16*>(part ? x.lo : x.hi) + static_cast<int64_t>(tok) * x.K +
                          (ch < 4 ? k0 : k1);
    st.c[i] = GLoad<U4>(src + 8 * (ch & 3));
  }
}

__device__ __forceinline__ void StoreA(const AStage& st, _Float16 (*As)[kTM][kARow], int m0, int M) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int idx = tid + i * kGT;
    const int part = idx >> 9, r = (idx >> 3) & 63, ch = idx & 7;
    const U4 v = m0 + r < M ? st.c[i] : U4{0u, 0u, 0u, 0u};
    *reinterpret_cast<U4*>(&As[part][r][8 * ch]) = v;
  }
}

// Byte-wise values v (0..255) of a dword as the f16 pairs (1024 + v0, 1024 +
// v2) and (1024 + v1, 1024 + v3), in the operand order of 4 inputs.
__device__ __forceinline__ void BytePairs(uint32_t v, H2* p02, H2* p13) {
  *p02 = AsH2((v & 0x00FF00FFu) | 0x64006400u);
  *p13 = AsH2(((v >> 8) & 0x00FF00FFu) | 0x64006400u);
}

__device__ __forceinline__ H8 Pack(H2 a, H2 b, H2 c, H2 d) {
  return __builtin_bit_cast(H8, U4{AsU(a), AsU(b), AsU(c), AsU(d)});
}

// Q8_0 weight operand of 8 int8 quants: (1024 + (q ^ 0x80)) - 1152 = q.
__device__ __forceinline__ H8 Q8Operand(U2 q) {
  const H2 off = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
  H2 p[4];
  BytePairs(q.x ^ 0x80808080u, &p[0], &p[1]);
  BytePairs(q.y ^ 0x80808080u, &p[2], &p[3]);
  return Pack(p[0] + off, p[1] + off, p[2] + off, p[3] + off);
}

__device__ __forceinline__ F4 Mfma32(H8 a, H8 b, F4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
// A fresh (zero-C) product: the empty asm keeps both sources live until the
// result exists, so the result is never allocated over a source -- an MFMA
// whose destination aliases its A or B registers returned wrong sums on
// gfx950 (measured), and the compiler allows it when a source dies there.
__device__ __forceinline__ F4 Mfma16Fresh(H4 a, H4 b) {
  const F4 r = __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, F4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  asm volatile("" ::"v"(a), "v"(b), "v"(r));
  return r;
}
// The same for a product accumulated onto c (c kept live too, so the result
// cannot partly overlap it either).
__device__ __forceinline__ F4 Mfma16Keep(H4 a, H4 b, F4 c) {
  const F4 r = __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  asm volatile("" ::"v"(a), "v"(b), "v"(c), "v"(r));
  return r;
}

// Q8_0 projections: a workgroup of 2 waves owns 64 tokens x 128 rows, each
// wave 64 x 64 = 4 x 4 MFMA tiles; a step covers one pair of 32-input blocks
// (K-step h = block h of the pair, scaled by its d once per K-step). The
// token operands of a step are staged in LDS for both waves; every lane
// assembles its weight operand from the raw quants; the next step's loads are
// in flight while the current one is multiplied.
__global__ __launch_bounds__(kGT) void QGemm8Kernel(GemmArgs a) {
  int nt = blockIdx.x, j = 0;
  while (j + 1 < a.n_jobs && nt >= a.tiles[j]) {
    nt -= a.tiles[j];
    ++j;
  }
  const GemmJob& J = a.job[j];
  // this split's block pairs [o0, o1)
  const int z = blockIdx.z, nall = a.x.K / 64;
  const int o0 = z * nall / a.ksplit, o1 = (z + 1) * nall / a.ksplit;
  const SplitX x = ShiftSplit(a.x, o0 * 64);
  const int m0 = blockIdx.y * kTM;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int jr = lane & 15, kq = lane >> 4;
  const int n0 = nt * kTN + wave * kWN;
  const int rows = J.w.rows;
  __shared__ __align__(16) _Float16 As[2][kTM][kARow];
  const uint8_t* wr[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
    wr[t] = J.w.w + static_cast<int64_t>(min(n0 + 16 * t + jr, rows - 1)) * J.w.row_bytes +
            static_cast<int64_t>(o0) * 68;
  struct Raw {
    U2 q0, q1;
    uint32_t d;
  };
  auto load_raw = [&](Raw& r, const uint8_t* pair) {
    r.q0 = GLoad<U2A2>(pair + 2 + 8 * kq);
    r.q1 = GLoad<U2A2>(pair + 36 + 8 * kq);
    r.d = static_cast<uint32_t>(GLoad<uint16_t>(pair)) | (static_cast<uint32_t>(GLoad<uint16_t>(pair + 34)) << 16);
  };
  const int nout = o1 - o0;
  F4 T[4][4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int t = 0; t < 4; ++t) T[mt][t] = F4{0.f, 0.f, 0.f, 0.f};
  AStage st;
  LoadA(st, x, m0, 0, 32);
  Raw raw[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) load_raw(raw[t], wr[t]);
  for (int o = 0; o < nout; ++o) {
    __syncthreads();
    StoreA(st, As, m0, x.M);
    __syncthreads();
    // the next pair's operands in flight during this one's products
    const int on = o + 1 < nout ? o + 1 : o;
    LoadA(st, x, m0, 64 * on, 64 * on + 32);
    Raw rn[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) load_raw(rn[t], wr[t] + 68 * on);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      H8 ah[4], al[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        ah[mt] = *reinterpret_cast<const H8*>(&As[0][16 * mt + jr][32 * h + 8 * kq]);
        al[mt] = *reinterpret_cast<const H8*>(&As[1][16 * mt + jr][32 * h + 8 * kq]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const H8 bf = Q8Operand(h ? raw[t].q1 : raw[t].q0);
        const float d = dev::HalfToFloatFast(h ? raw[t].d >> 16 : raw[t].d & 0xFFFFu);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
          const F4 c = Mfma32(al[mt], bf, Mfma32(ah[mt], bf, F4{0.f, 0.f, 0.f, 0.f}));
#pragma unroll
          for (int e = 0; e < 4; ++e) T[mt][t][e] = __builtin_fmaf(d, c[e], T[mt][t][e]);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) raw[t] = rn[t];
  }
  // epilogue: C[4*kq + e][jr] of each tile
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int tok = m0 + 16 * mt + 4 * kq + e;
      if (tok >= x.M) continue;
      const float is = x.inv_s[tok];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int row = n0 + 16 * t + jr;
        if (row >= rows) continue;
        PutOut(J, x, x.part, a.part_ld, a.pcol[j], a.ksplit, z, tok, row, T[mt][t][e] * is);
      }
    }
  }
}

// y = silu(g) * u elementwise, glibc-exact expf (reference src/kernels.h:82-92)
__global__ __launch_bounds__(256) void SwiGLUKernel(const float* __restrict__ g, const float* __restrict__ u,
                                                    float* __restrict__ y, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const float v = g[i];
  const float sg = v / __fadd_rn(1.0f, GlibcExpf(-v));
  y[i] = __fmul_rn(sg, u[i]);
}

}  // namespace

void SwiGLURows(const float* g, const float* u, float* y, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(SwiGLUKernel, dim3(static_cast<unsigned>(CeilDiv(n, 256))), dim3(256), 0, s, g, u, y, n);
  HIP_CHECK(hipGetLastError());
}

namespace {
// Floats of the split-K partials: tiled launches run at most this many partial
// tiles, two rounds of 256 compute units; up to 64 tokens, whose row tiles are
// few, one round (a session's first short segment allocates them).
constexpr int64_t PartTiles(int M) { return M <= 64 ? 256 : 512; }
int64_t PartFloats(int M, int n_max) {
  return std::max<int64_t>(PartTiles(M) * TiledTokens(M) * kTiledRows,
                           M < 96 ? static_cast<int64_t>(kGemmSplitMax) * M * n_max : 0);
}
}  // namespace

size_t SplitXBytes(int M, int K, int n_max) {
  const size_t big = static_cast<size_t>(M) * K * 2, small = static_cast<size_t>(M) * (K / 32) * 2;
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  return 2 * up(big) + 2 * up(small) + up(static_cast<size_t>(M) * 4) +
         up(static_cast<size_t>(PartFloats(M, n_max)) * 4);
}

SplitX SplitXView(void* base, int M, int K, int n_max) {
  const size_t big = static_cast<size_t>(M) * K * 2, small = static_cast<size_t>(M) * (K / 32) * 2;
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  uint8_t* p = static_cast<uint8_t*>(base);
  SplitX s;
  s.hi = p;
  s.lo = p + up(big);
  s.sum_hi = p + 2 * up(big);
  s.sum_lo = p + 2 * up(big) + up(small);
  s.inv_s = reinterpret_cast<float*>(p + 2 * up(big) + 2 * up(small));
  s.part = reinterpret_cast<float*>(p + 2 * up(big) + 2 * up(small) + up(static_cast<size_t>(M) * 4));
  s.part_floats = PartFloats(M, n_max);
  s.M = M;
  s.K = K;
  return s;
}

void SplitRowsAdd(float* X, int64_t ldx, int M, int K, const float* norm_w, float eps, const SplitX& out,
                  const SplitPending& pend, hipStream_t s) {
  RPG_CHECK(M > 0 && M <= out.M && K == out.K, "split rows: %d x %d does not fit the buffer", M, K);
  RPG_CHECK(K % 32 == 0 && K <= 8 * kSplitChunks * kSplitThreadsWide, "split rows: K = %d unsupported", K);
  RPG_CHECK(ldx % 4 == 0, "split rows: row stride must be a multiple of 4");
  RPG_CHECK(pend.part == nullptr || (pend.M == M && (pend.part_ld + pend.pcol) % 4 == 0 && pend.pcol % 4 == 0 &&
                                      pend.ksplit >= 1 && pend.ksplit <= kSplitPendMax),
            "split rows: pending sums do not match the rows");
  SplitX o = out;
  o.M = M;
  const dim3 grid(static_cast<unsigned>(M));
  const bool wide = K > 8 * kSplitChunks * kSplitThreads;
  const int nt = wide ? kSplitThreadsWide : kSplitThreads;
  const int nc = static_cast<int>(CeilDiv(K / 8, nt));
  const int variant =
      (norm_w != nullptr ? 1 : 0) + (pend.part == nullptr ? 0 : pend.ksplit <= kGemmSplitMax ? 2 : 4);
  auto launch = [&](auto nt_c, auto nc_c) {
    constexpr int NT = decltype(nt_c)::value, NC = decltype(nc_c)::value;
    constexpr int P4 = kGemmSplitMax, P8 = kSplitPendMax;
    const dim3 block(NT);
    switch (variant) {
      case 0: hipLaunchKernelGGL((SplitRowsKernel<NT, NC, false, 0>), grid, block, 0, s, X, ldx, K, norm_w, eps, o, pend); break;
      case 1: hipLaunchKernelGGL((SplitRowsKernel<NT, NC, true, 0>), grid, block, 0, s, X, ldx, K, norm_w, eps, o, pend); break;
      case 2: hipLaunchKernelGGL((SplitRowsKernel<NT, NC, false, P4>), grid, block, 0, s, X, ldx, K, norm_w, eps, o, pend); break;
      case 3: hipLaunchKernelGGL((SplitRowsKernel<NT, NC, true, P4>), grid, block, 0, s, X, ldx, K, norm_w, eps, o, pend); break;
      case 4: hipLaunchKernelGGL((SplitRowsKernel<NT, NC, false, P8>), grid, block, 0, s, X, ldx, K, norm_w, eps, o, pend); break;
      default: hipLaunchKernelGGL((SplitRowsKernel<NT, NC, true, P8>), grid, block, 0, s, X, ldx, K, norm_w, eps, o, pend);
    }
  };
  using N256 = std::integral_constant<int, kSplitThreads>;
  using N1024 = std::integral_constant<int, kSplitThreadsWide>;
  if (wide) {
    // 10240 < K <= 40960: two to five chunks per thread
    switch (nc) {
      case 2: launch(N1024{}, std::integral_constant<int, 2>{}); break;
      case 3: launch(N1024{}, std::integral_constant<int, 3>{}); break;
      case 4: launch(N1024{}, std::integral_constant<int, 4>{}); break;
      default: launch(N1024{}, std::integral_constant<int, kSplitChunks>{});
    }
  } else {
    switch (nc) {
      case 1: launch(N256{}, std::integral_constant<int, 1>{}); break;
      case 2: launch(N256{}, std::integral_constant<int, 2>{}); break;
      case 3: launch(N256{}, std::integral_constant<int, 3>{}); break;
      case 4: launch(N256{}, std::integral_constant<int, 4>{}); break;
      default: launch(N256{}, std::integral_constant<int, kSplitChunks>{});
    }
  }
  HIP_CHECK(hipGetLastError());
}

void SplitRows(const float* X, int64_t ldx, int M, int K, const float* norm_w, float eps, const SplitX& out,
               hipStream_t s) {
  // (no pending sums: the kernel does not write X)
  SplitRowsAdd(const_cast<float*>(X), ldx, M, K, norm_w, eps, out, SplitPending{}, s);
}

namespace {
// Whether the tiled kernel takes the matrix (its buffer resources and lane
// offsets are 32-bit).
bool TiledTakes(const MatRef& w) {
  return (w.type == kQ4_K || w.type == kQ6_K || w.type == kQ8_0) && w.cols % 256 == 0 &&
         w.row_bytes * w.rows < 0xFFFF0000LL;
}
}  // namespace

bool QGemmShares(const MatRef& a, const MatRef& b) {
  return a.type == b.type || (TiledMixes(a.type) && TiledMixes(b.type) && TiledTakes(a) && TiledTakes(b));
}

bool QGemmSupports(const MatRef& w) {
  return ((w.type == kQ4_K || w.type == kQ6_K) && TiledTakes(w)) || (w.type == kQ8_0 && w.cols % 64 == 0);
}

int ComputeUnits() {
  static int cached[64] = {};
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  RPG_CHECK(dev >= 0 && dev < 64, "device %d", dev);
  if (cached[dev] == 0) {
    int n = 0;
    HIP_CHECK(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    cached[dev] = n > 0 ? n : 1;
  }
  return cached[dev];
}

namespace {

// y = (y +) the sum of the split-K partials of one job, in split order.
__global__ __launch_bounds__(256) void SplitKReduceKernel(const float* __restrict__ part, int64_t part_ld, int pcol,
                                                          int ksplit, int M, int N, float* y, int64_t ldy, int epi) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<int64_t>(M) * N) return;
  const int tok = static_cast<int>(i / N), row = static_cast<int>(i % N);
  // every partial (and y) requested before the first is added: one round trip
  float* yp = y + static_cast<int64_t>(tok) * ldy + row;
  const float y0 = epi == kAdd ? *yp : 0.0f;
  float p[kTiledSplitMax];
#pragma unroll
  for (int z = 0; z < kTiledSplitMax; ++z)
    if (z < ksplit) p[z] = part[(static_cast<int64_t>(z) * M + tok) * part_ld + pcol + row];
  float v = 0.0f;
#pragma unroll
  for (int z = 0; z < kTiledSplitMax; ++z)
    if (z < ksplit) v += p[z];
  *yp = epi == kAdd ? y0 + v : v;
}

// K splits of a launch of `wgs` workgroups over `nblk` scale blocks: doubled
// while the launch has fewer than `target` workgroups, every split keeps at
// least `min_blk` blocks and the partials fit (thresholds measured on the
// Qwen3-4B projections at 512 tokens).
int ChooseSplit(int64_t wgs, int nblk, int64_t cols, const SplitX& x, int64_t target, int min_blk) {
  int S = 1;
  while (S < kGemmSplitMax && wgs * S < target && 2 * S * min_blk <= nblk &&
         static_cast<int64_t>(2 * S) * x.M * cols <= x.part_floats)
    S *= 2;
  return S;
}

// The K parts (1 .. kTiledSplitMax) of `wgs` tiled workgroups of `nblk`
// super-blocks on `cus` compute units (one tiled workgroup per unit): the
// count whose rounds of workgroups take the least time, a workgroup costing
// its super-blocks plus about 1.5 of pipeline fill and output (0.8 and 2.5
// measured the same). Every part keeps at least 1.67 super-blocks on average
// (2.5 left the 1.7B shapes 2 - 4 % slower at 128 - 512 tokens, 1 no faster
// than 1.67), and at most `max_parts` partial tiles are written.
int TiledParts(int64_t wgs, int nblk, int64_t cus, int64_t max_parts) {
  int best = 1;
  double best_cost = 0.0;
  for (int c = 1; c <= kTiledSplitMax; ++c) {
    if (c > 1 && (10 * c > 6 * nblk || c * wgs > max_parts)) break;
    const double cost = static_cast<double>(CeilDiv(c * wgs, cus)) * (static_cast<double>(nblk) / c + 1.5);
    if (c == 1 || cost < 0.95 * best_cost) best = c, best_cost = cost;
  }
  return best;
}

}  // namespace

void QGemm(const SplitX& x, const GemmJob* jobs, int n_jobs, hipStream_t s, SplitPending* defer, int cus) {
  RPG_CHECK(n_jobs >= 1 && n_jobs <= 3, "qgemm: 1..3 jobs");
  for (int j = 0; defer != nullptr && j < n_jobs; ++j) defer[j] = SplitPending{};
  int32_t pcol[3] = {0, 0, 0};
  int64_t cols = 0;
  for (int j = 0; j < n_jobs; ++j) {
    RPG_CHECK(QGemmSupports(jobs[j].w) && jobs[j].w.cols == x.K, "qgemm: unsupported matrix");
    RPG_CHECK(QGemmShares(jobs[j].w, jobs[0].w), "qgemm: types %u and %u in one launch", jobs[0].w.type, jobs[j].w.type);
    pcol[j] = static_cast<int32_t>(cols);
    cols += jobs[j].w.rows;
  }
  int S = 1;
  bool tiled = true;
  for (int j = 0; j < n_jobs; ++j) tiled = tiled && TiledTakes(jobs[j].w);
  if (tiled) {
    TiledArgs t;
    t.x = x;
    t.pair = 0;
    t.n_jobs = n_jobs;
    t.tokens = TiledTokens(x.M);
    t.tiles_m = static_cast<int32_t>(CeilDiv(x.M, t.tokens));
    int tiles = 0;
    for (int j = 0; j < n_jobs; ++j) {
      t.job[j] = jobs[j];
      t.tiles[j] = static_cast<int32_t>(CeilDiv(jobs[j].w.rows, kTiledRows));
      t.pcol[j] = pcol[j];
      tiles += t.tiles[j];
    }
    S = TiledParts(static_cast<int64_t>(tiles) * t.tiles_m, x.K / 256, cus > 0 ? cus : ComputeUnits(),
                   x.part_floats / (t.tokens * kTiledRows));
    while (S > 1 && static_cast<int64_t>(S) * x.M * cols > x.part_floats) --S;
    t.ksplit = S;
    t.part_ld = cols;
    LaunchTiled(t, s);
  } else {
    const int64_t mtiles = CeilDiv(x.M, kTM);
    GemmArgs a;
    a.x = x;
    a.n_jobs = n_jobs;
    int tiles = 0;
    for (int j = 0; j < n_jobs; ++j) {
      a.job[j] = jobs[j];
      a.tiles[j] = static_cast<int32_t>(CeilDiv(jobs[j].w.rows, kTN));
      a.pcol[j] = pcol[j];
      tiles += a.tiles[j];
    }
    const int nblk = x.K / 64;
    S = ChooseSplit(tiles * mtiles, nblk, cols, x, 320, 1);
    a.ksplit = S;
    a.part_ld = cols;
    const dim3 grid(static_cast<unsigned>(tiles), static_cast<unsigned>(mtiles), static_cast<unsigned>(S));
    hipLaunchKernelGGL(QGemm8Kernel, grid, dim3(kGT), 0, s, a);
  }
  HIP_CHECK(hipGetLastError());
  if (S > 1 && defer != nullptr) {
    for (int j = 0; j < n_jobs; ++j) {
      defer[j].part = x.part;
      defer[j].part_ld = cols;
      defer[j].pcol = pcol[j];
      defer[j].ksplit = S;
      defer[j].M = x.M;
    }
    return;
  }
  if (S > 1) {
    for (int j = 0; j < n_jobs; ++j) {
      const int64_t n = static_cast<int64_t>(x.M) * jobs[j].w.rows;
      hipLaunchKernelGGL(SplitKReduceKernel, dim3(static_cast<unsigned>(CeilDiv(n, 256))), dim3(256), 0, s, x.part,
                         cols, pcol[j], S, x.M, static_cast<int>(jobs[j].w.rows), jobs[j].y, jobs[j].ldy,
                         static_cast<int>(jobs[j].epi));
    }
    HIP_CHECK(hipGetLastError());
  }
}

void ApplyPending(const SplitPending& pend, float* y, int64_t ldy, int N, hipStream_t s, Epilogue epi) {
  if (pend.part == nullptr) return;
  RPG_CHECK(pend.ksplit >= 1 && pend.ksplit <= kTiledSplitMax, "pending sums: %d splits", pend.ksplit);
  const int64_t n = static_cast<int64_t>(pend.M) * N;
  hipLaunchKernelGGL(SplitKReduceKernel, dim3(static_cast<unsigned>(CeilDiv(n, 256))), dim3(256), 0, s, pend.part,
                     pend.part_ld, pend.pcol, pend.ksplit, pend.M, N, y, ldy, static_cast<int>(epi));
  HIP_CHECK(hipGetLastError());
}

bool QGemmSwiGLU(const SplitX& x, const GemmJob& gate, const GemmJob& up, hipStream_t s) {
  if (gate.w.type != up.w.type || gate.w.rows != up.w.rows || gate.w.cols != x.K || up.w.cols != x.K ||
      gate.w.row_bytes != up.w.row_bytes || x.K % 256 != 0)
    return false;
  if (!TiledTakes(gate.w) || !TiledTakes(up.w)) return false;
  TiledArgs t;
  t.x = x;
  t.pair = 1;
  t.n_jobs = 1;
  t.tokens = TiledTokens(x.M);
  t.tiles_m = static_cast<int32_t>(CeilDiv(x.M, t.tokens));
  t.job[0] = gate;
  t.job[1] = up;
  t.tiles[0] = static_cast<int32_t>(CeilDiv(gate.w.rows, kTiledRows / 2));
  t.tiles[1] = t.tiles[2] = 0;
  t.pcol[0] = t.pcol[1] = t.pcol[2] = 0;
  t.ksplit = 1;
  t.part_ld = 0;
  // The tiles past the last full round of compute units run in K parts, their
  // sums added by a second launch.
  const int64_t total = static_cast<int64_t>(t.tiles[0]) * t.tiles_m, cus = ComputeUnits(), tail = total % cus;
  t.tail_wg = static_cast<int32_t>(total - tail);
  t.tail_split = tail > 0 ? TiledParts(tail, x.K / 256, cus, x.part_floats / (t.tokens * kTiledRows)) : 1;
  LaunchTiled(t, s);
  return true;
}

}  // namespace k
}  // namespace rpg
