// Projections of a prompt's rows for gfx950: y[m, n] = sum_k x[m, k] W[n, k],
// bf16 operands, fp32 sums, for the row counts between the decode GEMVs (8
// rows) and the prompts that fill a library GEMM.
//
// Bound: the loads. W is read once per block of BM rows and x once per BN
// columns, and a CU has about 100 GB/s of LDS-DMA from its L2 and 25 GB/s of
// HBM: with the products left out the kernel takes the same time. So a
// workgroup walks K in stages of BK that arrive by LDS-DMA, DS - 1 stages
// ahead (40 to 112 KB in flight per workgroup, one or two of which fit a CU),
// with one barrier per stage, and the tile is chosen for the loads: as few rows
// as hold m, wide in n. (A CU's loads return in order: waves of their own for x,
// fetched less far ahead than W, waited just as long.)
//
// Products: v_mfma_f32_32x32x16_bf16, A = 32 rows of W, B = 32 rows of x, so
// that a lane ends with 4 neighbouring outputs of one row. LDS rows are
// xor-swizzled by 16-byte chunk (conflict-free b128 reads).
//
// Epilogues: bf16 rows; fp32 split-K partials [split, m, n] (where a few
// tiles would leave CUs idle: the residual add + RMSNorm sums them); SwiGLU
// (W blocks of 16 gate rows and the 16 up rows of the same columns, so that
// a lane holds both).
//
// Measured per launch in a graph over 600 MB of weights, beside the library GEMM
// (us; 16 / 64 / 128 / 256 / 512 rows; [n, k]; o and down with the planned splits):
//   o    [2560, 4096]   6.6 /  9.2 / 11.9 / 15.1 / 21.5    15.2 / 14.4 / 23.9 / 22.0 / 24.0
//   down [2560, 9728]  11.9 / 17.3 / 18.8 / 25.7 / 41.3    19.2 / 28.7 / 52.6 / 41.6 / 50.9
//   qkv  [6144, 2560]  15.3 / 19.0 / 19.1 / 24.2 / 37.2    12.3 / 16.1 / 19.1 / 31.3 / 27.6
//   gate/up [19456, 2560] with SwiGLU
//                      28.1 / 32.3 / 36.4 / 43.5 / 78.4    47.9 / 31.8 / 34.9 / 47.6 / 55.3, + 4 to 6 for silu_mul
// (In a 1 x 128 prefill under the kernel trace: o and down 16.2 on average, qkv
// 19.7, gate/up 35.1.) The row counts and sizes that take them: ek_kernels.py,
// linear_pays and its kin.

#include <atomic>
#include <cstring>

#include "ek_abi_internal.h"
#include "ek_attn_impl.h"
#include "ek_common.h"
#include "ek_hip.h"
#include "ek_hip_prompt.h"
#include "ek_lds_dma.h"

namespace {

enum { GE_BF16 = 0, GE_PARTS = 1, GE_SWIGLU = 2 };

struct GemmParams {
  const bf16_t* x; int64_t ldx;
  const bf16_t* w; int64_t ldw;
  bf16_t* y; int64_t ldy;
  float* parts;
  int m, n;            // output rows and columns (SwiGLU: gate columns)
  int stages;          // K stages
  int mt, nt;          // row and column tiles
};

// wait until at most n * PER of this wave's DMAs are outstanding: n stages ahead, 0 to
// 6 (DS - 2 at most), the same for the whole wave
template <int PER>
__device__ __forceinline__ void dma_wait(int n) {
#define EK_W(I) case I: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(I * PER < 63 ? I * PER : 63) : "memory"); break;
  switch (n) {
    EK_W(1) EK_W(2) EK_W(3) EK_W(4) EK_W(5) EK_W(6)
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
#undef EK_W
}

template <int BM, int BN, int BK, int NW, int DS>
struct GemmCfg {
  static constexpr int CH = BK / 8;                  // 16-byte chunks per LDS row
  static constexpr int RPI = 64 / CH;                // rows per DMA
  static constexpr int PW = BN / (RPI * NW);         // a wave's DMAs per stage: W rows
  static constexpr int PX = BM / (RPI * NW);         // and x rows
  static constexpr int WB = BN * BK * 2, XB = BM * BK * 2, SB = WB + XB;
  static constexpr int LDS = DS * SB;
  static constexpr int WM = BM / 32 < NW ? BM / 32 : NW;   // waves along m, the others along n
  static constexpr int WN = NW / WM;
  static constexpr int TM = BM / (32 * WM), TN = BN / (32 * WN);
  __device__ static int kx(int r) { return lds_xor<CH>(r); }
  static_assert(DS >= 3 && DS - 2 <= 6 && LDS <= 160 * 1024, "");   // dma_wait counts up to 6 stages
  static_assert(BN % (RPI * NW) == 0 && BM % (RPI * NW) == 0 && TM >= 1 && TN >= 1, "");
};

template <int EPI, int BM, int BN, int BK, int NW, int DS>
__global__ __launch_bounds__(64 * NW) void gemm_kernel(GemmParams p) {
  using C = GemmCfg<BM, BN, BK, NW, DS>;
  constexpr int TN = C::TN, TM = C::TM;
  extern __shared__ __align__(16) char lds[];
  const int lane = threadIdx.x & 63, w = wave_id();
  const int q = lane & 31, hh = lane >> 5;
  // tiles: the row blocks that share a W tile 8 ids apart (ids go round the 8 XCDs), column tiles in groups of 8
  int id = blockIdx.x;
  const int per = 8 * p.mt;
  const int grp = id / per;
  const int width = p.nt - 8 * grp < 8 ? p.nt - 8 * grp : 8;   // columns of this (the last) group
  id -= grp * per;
  const int mi = id / width, ni = 8 * grp + id % width;
  const int m0 = mi * BM, n0 = ni * (EPI == GE_SWIGLU ? BN / 2 : BN);
  const int sp = blockIdx.y;
  const int st0 = (int)((int64_t)p.stages * sp / (int)gridDim.y);             // this split's stages
  const int nst = (int)((int64_t)p.stages * (sp + 1) / (int)gridDim.y) - st0;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char_t*)lds;
  const char* wbase = reinterpret_cast<const char*>(p.w) + (int64_t)n0 * p.ldw * 2 + (int64_t)st0 * BK * 2;
  const char* xbase = reinterpret_cast<const char*>(p.x) + (int64_t)m0 * p.ldx * 2 + (int64_t)st0 * BK * 2;
  uint32_t wo[C::PW], xo[C::PX];
  const int srow = lane / C::CH, spos = lane % C::CH;
  // rows past the end re-read the last one (not stored)
#pragma unroll
  for (int j = 0; j < C::PW; ++j) {
    const int r = (j * NW + w) * C::RPI + srow;
    const int nr = p.n - n0;
    int64_t row;
    if (EPI == GE_SWIGLU) {   // a block of 32 rows: 16 gate rows, then the up rows of the same columns
      const int c = (r >> 5) * 16 + (r & 15);
      row = ((r & 16) ? (int64_t)p.n : 0) + (c < nr ? c : nr - 1);
    } else {
      row = r < nr ? r : nr - 1;
    }
    wo[j] = (uint32_t)(row * p.ldw * 2 + ((spos ^ C::kx(r)) * 16));
  }
#pragma unroll
  for (int j = 0; j < C::PX; ++j) {
    const int r = (j * NW + w) * C::RPI + srow;
    xo[j] = (uint32_t)((int64_t)(r < p.m - m0 ? r : p.m - m0 - 1) * p.ldx * 2 + ((spos ^ C::kx(r)) * 16));
  }
  // W where one row block holds all rows: non-temporal, no other workgroup reads
  // these bytes and x keeps the L2 (2 layers of a 1 x 128 prefill 223.8 -> 219.2
  // us; o and down at 4 rows, 4 layers and the head 429.4 -> 423.2)
  const bool once = p.mt == 1;
  auto fetch = [&](int st, int buf) {
    const uint32_t d = lds0 + buf * C::SB + w * 1024;
#pragma unroll
    for (int j = 0; j < C::PW; ++j) {
      if (once) lds_dma16_nt(d + j * NW * 1024, wbase + (int64_t)st * BK * 2, wo[j]);
      else lds_dma16(d + j * NW * 1024, wbase + (int64_t)st * BK * 2, wo[j]);
    }
#pragma unroll
    for (int j = 0; j < C::PX; ++j) lds_dma16(d + C::WB + j * NW * 1024, xbase + (int64_t)st * BK * 2, xo[j]);
  };
  for (int st = 0; st < DS - 1 && st < nst; ++st) fetch(st, st);
  const int wm = w % C::WM, wn = w / C::WM;

  int ra[BK / 16];            // LDS byte offset of this lane's operand chunk: row q of 32, chunk 2 i + hh
#pragma unroll
  for (int i = 0; i < BK / 16; ++i) ra[i] = q * BK * 2 + (((2 * i + hh) ^ C::kx(q)) * 16);
  f32x16_t acc[TM][TN];
#pragma unroll
  for (int u = 0; u < TM; ++u)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[u][t][e] = 0.f;

  int buf = 0, fb = DS - 1;
  for (int st = 0; st < nst; ++st) {
    const int ahead = nst - 1 - st;
    dma_wait<C::PW + C::PX>(ahead < DS - 2 ? ahead : DS - 2);
    // after the barrier stage st is in LDS and stage st - 1's reads are done: its buffer is free
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (st + DS - 1 < nst) {
      fetch(st + DS - 1, fb);
      fb = fb + 1 == DS ? 0 : fb + 1;
    }
    const lds_char_t* wp = (const lds_char_t*)lds + buf * C::SB + wn * TN * 32 * BK * 2;
    const lds_char_t* xp = (const lds_char_t*)lds + buf * C::SB + C::WB + wm * TM * 32 * BK * 2;
#pragma unroll
    for (int i = 0; i < BK / 16; ++i) {
      u32x4_t a[TN], b[TM];
#pragma unroll
      for (int u = 0; u < TM; ++u) b[u] = *(const lds_u32x4_t*)(xp + ra[i] + u * 32 * BK * 2);
#pragma unroll
      for (int t = 0; t < TN; ++t) a[t] = *(const lds_u32x4_t*)(wp + ra[i] + t * 32 * BK * 2);
#pragma unroll
      for (int u = 0; u < TM; ++u)
#pragma unroll
        for (int t = 0; t < TN; ++t)
          acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(eka::bf16x8_t, a[t]),
                                                           __builtin_bit_cast(eka::bf16x8_t, b[u]), acc[u][t], 0, 0, 0);
    }
    buf = buf + 1 == DS ? 0 : buf + 1;
  }

#pragma unroll
  for (int u = 0; u < TM; ++u) {
    const int m = m0 + 32 * (wm * TM + u) + q;
    if (m >= p.m) continue;
    if constexpr (EPI == GE_SWIGLU) {
      bf16_t* yr = p.y + (int64_t)m * p.ldy;
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const int n = n0 + 16 * (wn * TN + t) + 8 * a + 4 * hh;
          float o[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float g = rbf(acc[u][t][4 * a + c]), v = rbf(acc[u][t][8 + 4 * a + c]);
            o[c] = rbf(g / (1.0f + expf(-g))) * v;
          }
          if (n + 3 < p.n && ((reinterpret_cast<uintptr_t>(yr + n) & 7) == 0)) {
            *reinterpret_cast<uint2*>(yr + n) = make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
          } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
              if (n + c < p.n) yr[n + c] = (bf16_t)f2bf(o[c]);
          }
        }
    } else {
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const int n = n0 + 32 * (wn * TN + t) + 8 * a + 4 * hh;
          const f32x16_t& v = acc[u][t];
          if constexpr (EPI == GE_PARTS) {
            float* d = p.parts + ((int64_t)sp * p.m + m) * p.n + n;
            if (n + 3 < p.n && ((reinterpret_cast<uintptr_t>(d) & 15) == 0)) {
              *reinterpret_cast<float4*>(d) = make_float4(v[4 * a], v[4 * a + 1], v[4 * a + 2], v[4 * a + 3]);
            } else {
#pragma unroll
              for (int c = 0; c < 4; ++c)
                if (n + c < p.n) d[c] = v[4 * a + c];
            }
          } else {
            bf16_t* d = p.y + (int64_t)m * p.ldy + n;
            if (n + 3 < p.n && ((reinterpret_cast<uintptr_t>(d) & 7) == 0)) {
              *reinterpret_cast<uint2*>(d) = make_uint2(pack2(v[4 * a], v[4 * a + 1]), pack2(v[4 * a + 2], v[4 * a + 3]));
            } else {
#pragma unroll
              for (int c = 0; c < 4; ++c)
                if (n + c < p.n) d[c] = (bf16_t)f2bf(v[4 * a + c]);
            }
          }
        }
    }
  }
}

template <int EPI, int BM, int BN, int BK, int NW, int DS>
hipError_t launch(GemmParams p, int64_t k, int64_t sk, hipStream_t st) {
  using C = GemmCfg<BM, BN, BK, NW, DS>;
  auto fn = gemm_kernel<EPI, BM, BN, BK, NW, DS>;
  const int64_t stages = k / BK, bn = EPI == GE_SWIGLU ? BN / 2 : BN;
  const int64_t mt = (p.m + BM - 1) / BM, nt = (p.n + bn - 1) / bn;
  if (sk > stages || sk > 65535 || mt * nt > 0x7fffffff)
    return ek_fail(hipErrorInvalidValue, "linear: more splits than stages of 64, or too many tiles");
  p.stages = (int)stages;
  p.mt = (int)mt;
  p.nt = (int)nt;
  if (C::LDS > 64 * 1024) {   // per device: a kernel of more than 64 KB of LDS has to be allowed it
    static std::atomic<uint64_t> allowed{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 64 || !(allowed.load() >> dev & 1)) {
      e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
      if (e != hipSuccess) return e;
      if (dev < 64) allowed.fetch_or(1ull << dev);
    }
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)(mt * nt), (unsigned)sk), dim3(64 * NW), C::LDS, st, p);
  return hipGetLastError();
}

bool unaligned(const void* a) { return (reinterpret_cast<uintptr_t>(a) & 15) != 0; }

}  // namespace

bool ek_linear_takes(const void* x, const void* w, int64_t m, int64_t n, int64_t k, int64_t ldx, int64_t ldw) {
  // tile offsets are 32-bit: the up rows lie n rows from the gate rows, a tile is at most 256 rows
  return m >= 1 && n >= 1 && k >= 64 && k % 64 == 0 && m <= 0x7fffffff && n <= 0x3fffffff && !unaligned(x) &&
         !unaligned(w) && ldx >= 0 && ldw >= 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx < (1 << 22) && ldw < (1 << 22) &&
         (n + 256) * ldw * 2 < ((int64_t)1 << 32);
}

extern "C" {

int ek_linear(const void* x, const void* w, void* y, int64_t m, int64_t n, int64_t k, int64_t ldx, int64_t ldw,
              int64_t ldy, void* stream) {
  EK_GUARD();
  if (!ek_linear_takes(x, w, m, n, k, ldx, ldw))
    return ek_fail(hipErrorInvalidValue, "linear: K must be a multiple of 64, rows 16-byte aligned");
  GemmParams p;
  memset(&p, 0, sizeof(p));
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw;
  p.y = (bf16_t*)y; p.ldy = ldy; p.m = (int)m; p.n = (int)n;
  hipStream_t st = (hipStream_t)stream;
  // up to 32 rows the low tile; up to 128 the one of which two fit a CU (qkv at
  // 128 rows 17.6 us; 128-row tiles 20.6); up to 256 a wider one (21.8 us against
  // 28.3); beyond, 128 rows per tile (512 rows 37 against 44)
  if (m <= 32) return launch<GE_BF16, 32, 64, 64, 2, 6>(p, k, 1, st);
  if (m <= 128) return launch<GE_BF16, 64, 64, 64, 2, 4>(p, k, 1, st);
  if (m <= 256) return launch<GE_BF16, 64, 96, 64, 2, 3>(p, k, 1, st);
  return launch<GE_BF16, 128, 64, 64, 4, 3>(p, k, 1, st);
}

int ek_linear_parts(const void* x, const void* w, float* parts, int64_t m, int64_t n, int64_t k, int64_t ldx,
                    int64_t ldw, int64_t sk, void* stream) {
  EK_GUARD();
  if (!ek_linear_takes(x, w, m, n, k, ldx, ldw) || sk < 1)
    return ek_fail(hipErrorInvalidValue, "linear_parts: K must be a multiple of 64, rows 16-byte aligned");
  GemmParams p;
  memset(&p, 0, sizeof(p));
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw;
  p.parts = parts; p.m = (int)m; p.n = (int)n;
  hipStream_t st = (hipStream_t)stream;
  // at one workgroup per CU (the caller's sk): down at 64 rows 14.3 us on 64-row
  // tiles, 15.4 on 128; at 128 rows 17.9 on 128-row tiles, 20.6 on 64
  if (m <= 32) return launch<GE_PARTS, 32, 64, 64, 2, 6>(p, k, sk, st);
  if (m <= 64) return launch<GE_PARTS, 64, 64, 64, 2, 4>(p, k, sk, st);
  return launch<GE_PARTS, 128, 128, 64, 4, 4>(p, k, sk, st);
}

int ek_linear_swiglu(const void* x, const void* w, void* y, int64_t m, int64_t inter, int64_t k, int64_t ldx,
                     int64_t ldw, int64_t ldy, void* stream) {
  EK_GUARD();
  if (!ek_linear_takes(x, w, m, inter, k, ldx, ldw))
    return ek_fail(hipErrorInvalidValue, "linear_swiglu: K must be a multiple of 64, rows 16-byte aligned");
  GemmParams p;
  memset(&p, 0, sizeof(p));
  p.x = (const bf16_t*)x; p.ldx = ldx; p.w = (const bf16_t*)w; p.ldw = ldw;
  p.y = (bf16_t*)y; p.ldy = ldy; p.m = (int)m; p.n = (int)inter;
  hipStream_t st = (hipStream_t)stream;
  // tiles wide enough that the columns make one round over the CUs: gate/up
  // [19456, 2560] at 64 rows 28.4 us (128 columns 31.3), at 128 rows 34.1
  // (36.9), at 256 rows 41.3 (128 columns 65)
  if (m <= 32) return launch<GE_SWIGLU, 32, 128, 64, 2, 4>(p, k, 1, st);
  if (m <= 64) return launch<GE_SWIGLU, 64, 96, 64, 2, 3>(p, k, 1, st);
  if (m <= 128) return launch<GE_SWIGLU, 128, 96, 64, 4, 5>(p, k, 1, st);
  return launch<GE_SWIGLU, 128, 160, 64, 4, 4>(p, k, 1, st);
}

}  // extern "C"
