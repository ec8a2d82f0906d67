// Prefill attention for gfx950: causal GQA flash attention over the prompt's
// keys, on the matrix cores. The reference runs torch SDPA here
// (engine/ek_model.py:315-323) with the prompt's additive mask: key <= query
// and key >= start[b] (left padding, engine.py:541-570); query rows with no
// visible key (the padding rows) attend to themselves, as this build's torch
// path does, so that their K/V rows stay finite (no decode step reads them).
//
// The same kernel scores a speculative verify step (ek_attn_verify; the
// reference's flash_verify, engine/ek_kernels.py:1419, restated by its torch
// fallback attn_torch, :1451): the row's S query tokens then sit at cache
// positions q0[b] .. q0[b] + S - 1 (after the row's cached keys), query j
// sees keys [start[b], q0[b] + j].
//
// attn_flash_kernel runs both: whole rows (4 waves share each K/V tile), or,
// for a verify step, one wave per share of the row's keys and a second launch
// that combines the shares.

#include <atomic>
#include <cstring>

#include "ek_abi_internal.h"
#include "ek_attn_impl.h"
#include "ek_common.h"
#include "ek_hip.h"
#include "ek_lds_dma.h"

namespace {

constexpr int KB = 32;   // a split's keys are a multiple of this

struct PrefillParams {
  const bf16_t* q; int64_t ldq;       // q of token t, head j: q + (b * S + t) * ldq + j * D
  const bf16_t* kc; const bf16_t* vc; int64_t csb, csh, css;
  const int32_t* start;               // [B] first visible key (left padding)
  const int64_t* q0;                  // [B] cache position of query token 0 (verify), or null (prefill: 0)
  bf16_t* out; int64_t ldo;           // out row (b * S + t), head j at j * D
  int64_t s;                          // query tokens per row (prefill: the padded prompt length)
  int64_t s_cap;                      // cache rows per (batch row, kv head)
  int nkv;
  float scale;
  // key splits (verify): split sp of a query block takes keys [k0 + sp * kchunk,
  // + kchunk) and writes its unnormalised output and (max, sum) to po / pml
  int nsplit;                         // 1: no split, the normalised output goes to out
  int64_t kchunk;                     // keys per split (a multiple of KB)
  float* po;                          // [nsplit][B*S][n_q][D]
  float* pml;                         // [nsplit][B*S][n_q][2]
  int nq;                             // query heads (n_kv * G)
  int nb, qlast;                      // batch rows; the launch's last query block (attn_flash_kernel)
  int64_t row0;                       // the launch's first row (attn_split_combine_kernel)
};

// ---------------------------------------------------------------------------
// The prompt's attention (one split)
// ---------------------------------------------------------------------------
// this wave's loads into LDS have landed and its LDS reads are done: of the
// other buffer, which is filled next. (One wave per workgroup has no barrier
// that would wait for the reads.)
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

// The schedule of N products, each of R LDS reads: the reads of AHEAD products
// first, then a product and the next one's reads in turn (left to itself the
// compiler reads each operand right before its product and waits for it:
// 1 x 16000 tokens 1.90 -> 1.86 ms, 4 x 777 24.0 -> 22.3 us, both sides with a
// running maximum that moved past a growth of 2^4).
template <int N, int AHEAD, int R>
__device__ __forceinline__ void sched_ahead() {
  constexpr int A = AHEAD < N ? AHEAD : N;
  __builtin_amdgcn_sched_group_barrier(0x100, A * R, 0);
#pragma unroll
  for (int i = 0; i < N - A; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, R, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, A, 0);
}

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

// 8 neighbouring values of a product's result as bf16
__device__ __forceinline__ uint4 pack8(const f32x16_t& v, int e) {
  return make_uint4(pack2(v[e], v[e + 1]), pack2(v[e + 2], v[e + 3]), pack2(v[e + 4], v[e + 5]), pack2(v[e + 6], v[e + 7]));
}

constexpr int FKT = 64;      // keys per tile
constexpr int FNWV = 4;      // waves per workgroup (whole rows)

// One tile of K (or V) in LDS: FKT rows of D bf16, row-major, the 16-byte
// chunks of row r permuted by an xor. K is read a chunk column at a time
// (ds_read_b128, 32 rows): rows that share banks differ in kx. V is read
// through ds_read_b64_tr_b16 (4 rows x 64 bytes per half wave): vx moves the
// 64-byte blocks of the 4 rows to different banks.
template <int D, int NW>
struct FlTile {
  static constexpr int CH = D / 8;                   // chunks per row
  static constexpr int RPI = 64 / CH;                // rows one wave's DMA brings
  static constexpr int NI = FKT / (RPI * NW);        // DMAs per wave and tile
  static constexpr int BYTES = FKT * D * 2;
  __device__ static int kx(int r) { return lds_xor<CH>(r); }
  __device__ static int vx(int r) { return D == 128 ? (r & 3) << 2 : D == 64 ? (r & 2) << 1 : 0; }
};

// Bound: the matrix cores. A wave holds 32 query rows of one head and walks
// the keys in tiles of FKT that the workgroup's 4 waves share through LDS:
//
//   S^T[64 keys x 32 q] = K . Q^T      v_mfma_f32_32x32x16_bf16, the query in
//                                      the lane: its max and sum stay there,
//                                      one half-wave swap per tile
//   O^T[D x 32 q] += V^T . P^T         P^T straight from S^T's registers: lane
//                                      (q, h) holds keys 8 a + 4 h + c, and V's
//                                      rows are read in that key order
//
// K/V tiles arrive by LDS-DMA, double-buffered, one barrier per tile; V is
// transposed by the read. The running max is exact and O is rescaled in every
// tile in which one of the wave's rows finds a larger one: the heaviest weight of
// a tile is then 1 and the next ones lie just below it, where bf16 is finest. The
// row's sum takes the weights as the value products do, rounded, so that their
// common part cancels. Error against 64 bits (N(0, 1) inputs, 32/8 heads, D 128;
// this / a maximum per 32 keys and sums of unrounded weights): 1 x 16000 tokens
// 2.081e-3 / 2.083e-3, 1 x 3000 2.025e-3 / 2.029e-3, 1 x 100 1.849e-3 / 1.865e-3.
// A maximum that moves only past a growth of 2^4 takes 5 to 7 % less time (1 x
// 16000 tokens 1.88 against 1.98 ms, 4 x 777 22.6 against 24.4 us, one card) and
// leaves 2.151e-3 and 2.099e-3. Two workgroups per CU: one's softmax runs beside
// the other's products.
//
// P2 (a verify step's tokens): each weight goes through the value products as
// two bf16 parts, its rounding and what that leaves, so that the result's own
// rounding is the only one that counts (3 tokens over 2100 keys 1.66e-3; one part
// and a maximum per 64 keys of a split 2.10e-3, per 32 keys 2.08e-3; 15.4 -> 16.0
// us, the tiles are few). Prompts, bound by these products, take one part.
//
// SPLIT (a verify step's few tokens over many keys): a workgroup is one wave,
// its 32 query columns are (token, head) pairs of one kv head (column c: token
// c / G, head c % G), its keys one of p.nsplit shares of the row; it leaves its
// unnormalised rows and their (max in log2, sum) to the combine. Bound: the
// two launches and one K/V tile's round trip. Measured (1 x 3 tokens, 2100
// keys, 32/8 heads, D 128, with the combine): 15.5 us, where a workgroup of 16
// query columns per head, mostly empty, and the serial combine took 29.6.
//
// KG = 2: two groups of 4 waves take a row block's tiles in turn, each with
// its own buffers, and merge at the end through LDS. One workgroup per CU
// then has the two waves per SIMD that two workgroups have otherwise, and the
// longest block half as many tiles: for launches that leave CUs empty.
// Measured (us, KG 1 / 2): 32/8 heads, D 128: 1 x 256 tokens 10.6 / 11.1, 1 x 512
// 16.0 / 15.2, 1 x 1024 26.9 / 23.9; 16/8 heads 1 x 2048 45.9 / 37.8; 8/8 heads,
// D 64, 1 x 2048 32.0 / 24.9; 1 x 128 8.0 / 8.9.
template <int D, int G, bool SPLIT, int KG, bool P2>
__global__ __launch_bounds__(64 * (SPLIT ? 1 : FNWV * KG), SPLIT ? 1 : 2) void attn_flash_kernel(PrefillParams p) {
  constexpr int NW = SPLIT ? 1 : FNWV;               // waves that share a tile
  using T = FlTile<D, NW>;
  constexpr int HG = SPLIT ? G : (G < FNWV ? G : FNWV);      // heads of a workgroup
  constexpr int HS = G / HG;                                 // workgroups that share a kv head's group
  constexpr int TB = SPLIT ? 32 / G : 32 * (FNWV / HG);      // query tokens of a workgroup
  constexpr int KS = D / 16;                         // k-steps of QK^T
  constexpr int DB = D / 32;                         // 32-dim blocks of O
  static_assert(KG == 1 || !(SPLIT || P2), "");
  extern __shared__ __align__(16) char lds_all[];    // per key group: [buffer][K, V]

  const int tid = threadIdx.x, lane = tid & 63;
  const int kg = KG == 1 ? 0 : wave_id() / NW, w = KG == 1 ? wave_id() : wave_id() - kg * NW;
  char* lds = lds_all + kg * 4 * T::BYTES;
  const int q = lane & 31, hh = lane >> 5;
  // blocks in launch order: kv head fastest (blocks go round the XCDs: with 8 kv
  // heads an XCD's L2 holds one head's keys), the longest query blocks first
  const int units = p.nkv * HS;
  const int hu = SPLIT ? blockIdx.x % units : blockIdx.x;
  const int sp = SPLIT ? blockIdx.x / units : 0;
  const int b = blockIdx.y;
  const int qblk = p.qlast - (int)blockIdx.z;
  const int h = hu / HS;
  const int head = h * G + (SPLIT ? q % G : (hu % HS) * HG + (w % HG));
  const int s = (int)p.s;
  int64_t qb64 = p.q0 ? p.q0[b] : 0;
  qb64 = qb64 < 0 ? 0 : (qb64 > p.s_cap - p.s ? p.s_cap - p.s : qb64);
  const int qb = (int)qb64;                          // cache position of query token 0
  const int kend = qb + s;
  int pad = p.start[b];
  pad = pad < 0 ? 0 : (pad > kend ? kend : pad);
  const int t0 = qblk * TB;                          // the workgroup's tokens [t0, tend)
  const int tend = t0 + TB < s ? t0 + TB : s;
  int k0 = qb + t0 < pad ? qb + t0 : pad;            // its keys [k0, k1)
  int k1 = qb + tend;
  if (SPLIT) {
    const int64_t a = k0 + sp * p.kchunk, e = a + p.kchunk;
    k0 = a < k1 ? (int)a : k1;
    k1 = e < k1 ? (int)e : k1;
  }
  // A masked key's weight is 0, but 0 times a value that is not finite is not: a
  // tile's keys past a token would reach it. Rows past k1 and before klo are
  // re-reads, and where a workgroup has several 32-token blocks (HG < 4) tiles
  // start at a block and a half past a wave's last token takes the other half's
  // values, so that a value row reaches at most 31 tokens back (a prompt's; a
  // verify step's tokens are few). 4 x 777 tokens, 16/8 heads: 24.4 -> 24.7 us
  // (skipping that half's products instead: 25.3).
  constexpr bool CUT = !SPLIT && HG < FNWV;
  const int klo = k0;
  if (CUT && !p.q0) k0 &= ~31;
  const int ntile = (k1 - k0 + FKT - 1) / FKT;
  constexpr int TW = SPLIT ? TB : 32;                // tokens of a wave
  const int tw = SPLIT ? t0 : t0 + 32 * (w / HG);    // this wave's first token
  const int tl = tw + (SPLIT ? q / G : q);           // this lane's token
  const int tok_r = tl < s ? tl : s - 1;             // (past the prompt: its last, not stored)
  const int tok = qb + tok_r;                        // its cache position
  const int tmin = qb + (tw < s ? tw : s - 1);
  const int tmax = qb + (tw + TW - 1 < s ? tw + TW - 1 : s - 1);

  const char* kb = reinterpret_cast<const char*>(p.kc + b * p.csb + h * p.csh);
  const char* vb = reinterpret_cast<const char*>(p.vc + b * p.csb + h * p.csh);
  const int64_t rowb = p.css * 2;                    // bytes of a cache row
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int srow = lane / T::CH, spos = lane % T::CH;    // this lane's place in a DMA
  // a DMA's first row r0 is a multiple of RPI: kx(r0 + srow) = kx(r0) ^ kx(srow), vx(r0 + srow) = vx(srow)
  const int kch = (spos ^ T::kx(srow)) * 16, vch = (spos ^ T::vx(srow)) * 16;
  const bool wide = p.css >= ((int64_t)1 << 26);     // rows beyond 32-bit offsets: 64-bit addresses throughout
  const uint32_t rvo = wide ? 0u : (uint32_t)(srow * rowb);
  const uint32_t kvo = rvo + (kch ^ (T::kx(w * T::RPI) * 16)), vvo = rvo + vch;   // NW > 1: kx(r0) is the wave's
  auto stage = [&](int buf, int kt) {
    const uint32_t kl = lds0 + buf * 2 * T::BYTES, vl = kl + T::BYTES;
    if (kt + FKT <= k1 && !wide && (!CUT || kt >= klo)) {
#pragma unroll
      for (int j = 0; j < T::NI; ++j) {
        const int r0 = (j * NW + w) * T::RPI;
        lds_dma16(kl + r0 * D * 2, kb + (kt + r0) * rowb, NW > 1 ? kvo : rvo + (kch ^ (T::kx(r0) * 16)));
        lds_dma16(vl + r0 * D * 2, vb + (kt + r0) * rowb, vvo);
      }
    } else {   // rows past the last key re-read it, rows before the first that one (masked below)
#pragma unroll
      for (int j = 0; j < T::NI; ++j) {
        const int r0 = (j * NW + w) * T::RPI;
        int key = kt + r0 + srow;
        key = key < k1 ? key : k1 - 1;
        if (CUT) key = key < klo ? klo : key;
        lds_dma16_addr(kl + r0 * D * 2, kb + key * rowb + (kch ^ (T::kx(r0) * 16)));
        lds_dma16_addr(vl + r0 * D * 2, vb + key * rowb + vch);
      }
    }
  };
  if (kg < ntile) stage(0, k0 + kg * FKT);

  // this lane's query row, the B operand of QK^T; a negative scale goes into its signs
  uint4 qf[KS];
  // weights are 2^(sc2 (s - m)); at scale 0 small but not 0, so that a masked -inf stays one
  const float sc2 = p.scale == 0.f ? 1e-37f : fabsf(p.scale) * 1.44269504088896341f;
  {
    const bf16_t* qrow = p.q + ((int64_t)b * p.s + tok_r) * p.ldq + (int64_t)head * D + 8 * hh;
    const uint32_t flip = p.scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      qf[i] = ld16(qrow + 16 * i);
      qf[i].x ^= flip; qf[i].y ^= flip; qf[i].z ^= flip; qf[i].w ^= flip;
    }
  }
  // LDS byte offsets: K row q (of 32), chunk 2 i + hh; V row 4 hh + (lane & 15) / 4, dims 16 ((lane >> 4) & 1) + 4 (lane & 3)
  int ka[KS], va[DB];
#pragma unroll
  for (int i = 0; i < KS; ++i) ka[i] = q * D * 2 + (((2 * i + hh) ^ T::kx(q)) * 16);
  {
    const int vr = (lane & 15) >> 2, i4 = lane & 3;
#pragma unroll
    for (int j = 0; j < DB; ++j)
      va[j] = (4 * hh + vr) * D * 2 + (((4 * j + 2 * ((lane >> 4) & 1) + (i4 >> 1)) ^ T::vx(vr)) * 16) + (i4 & 1) * 8;
  }

  f32x16_t o[DB];
#pragma unroll
  for (int j = 0; j < DB; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[j][e] = 0.f;
  float m = -1e30f, l = 0.f;
  const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);

  for (int i0 = 0; i0 < ntile; i0 += KG) {           // group kg: tiles kg, kg + KG, ...
    const int it = i0 + kg, buf = (i0 / KG) & 1;
    const int kt = k0 + it * FKT;
    dma_wait();
    __syncthreads();      // tile `it` is in LDS; the other buffer is no longer read
    if (it + KG < ntile) stage(buf ^ 1, kt + KG * FKT);
    if (it >= ntile || kt > tmax) continue;          // no tile left, or past this wave's tokens
    const __attribute__((address_space(3))) char* kl =
        (const __attribute__((address_space(3))) char*)lds + buf * 2 * T::BYTES;
    f32x16_t sv[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int e = 0; e < 16; ++e) sv[kk][e] = 0.f;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const u32x4_t kf = *(const lds_u32x4_t*)(kl + ka[i] + kk * 32 * D * 2);
        sv[kk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(eka::bf16x8_t, kf), eka::as_bf16x8(qf[i]),
                                                         sv[kk], 0, 0, 0);
      }
    }
    sched_ahead<2 * KS, 6, 1>();   // 4 to 10 reads ahead measured the same; on the value products: no gain
    if (kt + FKT - 1 > tmin || kt < pad || (SPLIT && kt + FKT > k1)) {   // the diagonal, the last key, or padding
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = kt + 32 * kk + 8 * (e >> 2) + 4 * hh + (e & 3);
          const bool ok = ((key <= tok && key >= pad) || (tok < pad && key == tok)) && (!SPLIT || key < k1);
          sv[kk][e] = ok ? sv[kk][e] : -INFINITY;
        }
    }
    float mx = sv[0][0];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sv[kk][e]);
    {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float a = __builtin_amdgcn_exp2f((m - mn) * sc2);
      m = mn;
      l *= a;
#pragma unroll
      for (int j = 0; j < DB; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[j][e] *= a;
    }
    const float mc = m * sc2;
    uint4 pf[2][2], pl[2][2];                        // the weights' bf16 parts (pl: P2)
    float ls[2] = {0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        sv[kk][e] = __builtin_amdgcn_exp2f(fmaf(sv[kk][e], sc2, -mc));
        if (P2) ls[kk] += sv[kk][e];
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        pf[kk][j] = pack8(sv[kk], 8 * j);
        if constexpr (P2) {
          float hi[8];
          unpack8(pf[kk][j], hi);
#pragma unroll
          for (int e = 0; e < 8; ++e) sv[kk][8 * j + e] -= hi[e];
          pl[kk][j] = pack8(sv[kk], 8 * j);
        } else {
          ls[kk] = dot8_acc_d2(pf[kk][j], ones, ls[kk]);
        }
      }
    }
    l += ls[0] + ls[1];
    // past the wave's last token the weights are 0: the first half's values again
    const __attribute__((address_space(3))) char* vl1 = CUT && kt + 32 > tmax ? kl - 32 * D * 2 : kl;
    // O^T: the A operand of k-step (kk, j) is V^T of keys 32 kk + 16 j + 4 hh + {0..3, 8..11}
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          const __attribute__((address_space(3))) char* vl = (kk ? vl1 : kl) + T::BYTES + va[d] + (32 * kk + 16 * j) * D * 2;
          const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)vl);
          const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vl + 8 * D * 2));
          const auto vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(eka::bf16x8_t, vf),
                                                         eka::as_bf16x8(pf[kk][j]), o[d], 0, 0, 0);
          if constexpr (P2)
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(eka::bf16x8_t, vf),
                                                           eka::as_bf16x8(pl[kk][j]), o[d], 0, 0, 0);
        }
  }
  {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  if constexpr (KG > 1) {   // group 0 takes in the others' rows: lane for lane, 4 dims at a time
    __syncthreads();                                 // the tiles are no longer read
    float* ex = reinterpret_cast<float*>(lds_all) + (size_t)w * 64 * (DB * 16 + 2) + lane;
    if (kg == 1) {
      ex[0] = m;
      ex[64] = l;
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) ex[64 * (2 + 16 * d + e)] = o[d][e];
    }
    __syncthreads();
    if (kg == 1) return;
    const float m1 = ex[0], mn = fmaxf(m, m1);
    const float a0 = __builtin_amdgcn_exp2f((m - mn) * sc2), a1 = __builtin_amdgcn_exp2f((m1 - mn) * sc2);
    l = l * a0 + ex[64] * a1;
    m = mn;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[d][e] = o[d][e] * a0 + ex[64 * (2 + 16 * d + e)] * a1;
  }
  if (tl >= s) return;
  if constexpr (SPLIT) {
    const int64_t idx = ((int64_t)sp * p.nb * s + (int64_t)b * s + tl) * p.nq + head;
    if (hh == 0) {
      p.pml[2 * idx] = m * sc2;
      p.pml[2 * idx + 1] = l;
    }
    if (ntile == 0) return;
    float* prow = p.po + idx * D + 4 * hh;
    const bool pal = (reinterpret_cast<uintptr_t>(p.po) & 15) == 0;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int a = 0; a < 4; ++a) {   // dims 32 d + 8 a + 4 hh + 0..3
        float* dst = prow + 32 * d + 8 * a;
        if (pal) {
          *reinterpret_cast<float4*>(dst) = make_float4(o[d][4 * a], o[d][4 * a + 1], o[d][4 * a + 2], o[d][4 * a + 3]);
        } else {
          dst[0] = o[d][4 * a]; dst[1] = o[d][4 * a + 1]; dst[2] = o[d][4 * a + 2]; dst[3] = o[d][4 * a + 3];
        }
      }
    return;
  }
  const float inv = l > 0.f ? __builtin_amdgcn_rcpf(l) : 0.f;   // to 1 ulp of fp32; the result is rounded to bf16
  bf16_t* orow = p.out + ((int64_t)b * p.s + tok_r) * p.ldo + (int64_t)head * D + 4 * hh;
  const bool al = (reinterpret_cast<uintptr_t>(p.out) & 7) == 0;   // rows are 16-byte multiples apart
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int a = 0; a < 4; ++a) {   // dims 32 d + 8 a + 4 hh + 0..3
      const float x0 = o[d][4 * a] * inv, x1 = o[d][4 * a + 1] * inv, x2 = o[d][4 * a + 2] * inv, x3 = o[d][4 * a + 3] * inv;
      bf16_t* dst = orow + 32 * d + 8 * a;
      if (al) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(pack2(x0, x1), pack2(x2, x3));
      } else {
        dst[0] = (bf16_t)f2bf(x0); dst[1] = (bf16_t)f2bf(x1); dst[2] = (bf16_t)f2bf(x2); dst[3] = (bf16_t)f2bf(x3);
      }
    }
}

// The key splits' rows combined: out = sum_s o_s 2^(m_s - M) / sum_s l_s
// 2^(m_s - M), rounded to bf16 once. One workgroup per (query row, head): a
// group of D / 4 lanes per split, four splits' loads in flight per lane, the
// groups' sums added through LDS (4.8 us for 32 splits of 3 rows x 32 heads; a
// thread walking the splits one after another, a load round trip each, 15.6).
template <int D>
__global__ __launch_bounds__(256) void attn_split_combine_kernel(PrefillParams p) {
  constexpr int LP = D / 4, NGR = 256 / LP;
  __shared__ float wgt[256], lw[256], red[NGR][D];
  const int64_t row = p.row0 + blockIdx.x, head = blockIdx.y, rows = p.nb * p.s;
  const int tid = threadIdx.x, g = tid / LP, c = tid % LP;
  float ms = -INFINITY, ls = 0.f;
  if (tid < p.nsplit) {
    const int64_t idx = (tid * rows + row) * p.nq + head;
    ms = p.pml[2 * idx];
    ls = p.pml[2 * idx + 1];
    if (ls == 0.f) ms = -INFINITY;        // a split without keys: its row was not written
  }
  // the first round of rows loads while the weights are made
  float v[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int sp = g + i * NGR;
    sp = sp < p.nsplit ? sp : p.nsplit - 1;
    const float* src = p.po + ((sp * rows + row) * p.nq + head) * D + c;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[i][k] = src[k * LP];
  }
  wgt[tid] = ms;
  lw[tid] = ls;
  __syncthreads();
  float mx = -INFINITY, l = 0.f;
  for (int s = 0; s < p.nsplit; ++s) mx = fmaxf(mx, wgt[s]);
  for (int s = 0; s < p.nsplit; ++s) l += wgt[s] > -INFINITY ? lw[s] * __builtin_amdgcn_exp2f(wgt[s] - mx) : 0.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < p.nsplit; s0 += 4 * NGR) {
    if (s0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int sp = s0 + g + i * NGR;
        sp = sp < p.nsplit ? sp : p.nsplit - 1;
        const float* src = p.po + ((sp * rows + row) * p.nq + head) * D + c;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[i][k] = src[k * LP];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int sp = s0 + g + i * NGR;
      if (sp >= p.nsplit || !(wgt[sp] > -INFINITY)) continue;
      const float w = __builtin_amdgcn_exp2f(wgt[sp] - mx);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] = fmaf(v[i][k], w, acc[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) red[g][c + k * LP] = acc[k];
  __syncthreads();
  if (tid < D) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NGR; ++i) t += red[i][tid];
    p.out[row * p.ldo + head * D + tid] = (bf16_t)f2bf(l == 0.f ? 0.f : t / l);   // a NaN row stays NaN
  }
}

// compute units of the current device (256 on MI355X)
int cu_count() {
  static std::atomic<int> cache[64];
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if ((n = cache[dev].load()) > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
  cache[dev].store(n);
  return n;
}

template <int D, int G>
hipError_t launch_prefill(const PrefillParams& p, int64_t b, hipStream_t st) {
  const bool split = p.nsplit > 1;
  constexpr int HG = G < FNWV ? G : FNWV;
  const int tb = split ? 32 / G : 32 * (FNWV / HG);      // query tokens of a workgroup
  PrefillParams f = p;
  f.nb = (int)b;
  const int64_t nqb = (p.s + tb - 1) / tb;
  const int64_t x = (int64_t)p.nkv * (split ? p.nsplit : G / HG), blocks = nqb * b * x;
  constexpr int LDS = 4 * FKT * D * 2;                   // two buffers of K and V
  void (*fn)(PrefillParams) = attn_flash_kernel<D, G, false, 1, false>;
  int threads = 64 * FNWV, lds = LDS;
  if (split) {
    fn = attn_flash_kernel<D, G, true, 1, true>;
    threads = 64;
  } else if (p.q0 && p.s_cap <= 256) {
    // a verify step whose cache takes no split (verify_splits): few keys, the launch counts
    fn = attn_flash_kernel<D, G, false, 1, true>;
  } else if (blocks <= cu_count() && p.s > 4 * FKT) {
    // fewer workgroups than CUs, and rows long enough to pay for the merge: two key groups each
    fn = attn_flash_kernel<D, G, false, 2, false>;
    threads *= 2;
    lds *= 2;
    if (lds > 64 * 1024) {   // more LDS than a kernel has by default
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return e;
    }
  }
  // a grid of at most 65535 query blocks (y, z); x threads stay below 2^32
  for (int64_t z0 = 0; z0 < nqb; z0 += 65535) {
    const int64_t nz = nqb - z0 < 65535 ? nqb - z0 : 65535;
    f.qlast = (int)(nqb - 1 - z0);
    hipLaunchKernelGGL(fn, dim3((unsigned)x, (unsigned)b, (unsigned)nz), dim3(threads), lds, st, f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (!split) return hipSuccess;
  for (f.row0 = 0; f.row0 < b * p.s; f.row0 += 0xffffff) {   // 2^32 threads along x
    const int64_t nr = b * p.s - f.row0 < 0xffffff ? b * p.s - f.row0 : 0xffffff;
    hipLaunchKernelGGL((attn_split_combine_kernel<D>), dim3((unsigned)nr, (unsigned)p.nq), dim3(256), 0, st, f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int D>
hipError_t launch_prefill_g(const PrefillParams& p, int g, int64_t b, hipStream_t st) {
  switch (g) {
    case 1: return launch_prefill<D, 1>(p, b, st);
    case 2: return launch_prefill<D, 2>(p, b, st);
    case 4: return launch_prefill<D, 4>(p, b, st);
    case 8: return launch_prefill<D, 8>(p, b, st);
    default: return ek_fail(hipErrorInvalidValue, "attn_prefill: query heads per kv head must be 1, 2, 4 or 8");
  }
}

}  // namespace

namespace {

hipError_t attn_flash(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, int64_t csb, int64_t csh,
                      int64_t css, int64_t s_cap, const int32_t* start, const int64_t* q0, void* out, int64_t ldo,
                      int64_t b, int64_t s, int64_t n_q, int64_t n_kv, int64_t head_dim, float sm_scale,
                      void* stream, float* part = nullptr, int64_t part_floats = 0, int64_t splits = 1) {
  if (b < 1 || b > 65535 || s < 1 || s > s_cap || n_kv < 1 || n_kv > 65535 || n_q % n_kv)
    return ek_fail(hipErrorInvalidValue, "attn_prefill/attn_verify: bad batch, length or head counts");
  // (the second limit is the entry points' own, in blocks of 16 tokens: no kernel here needs it)
  if (splits < 1 || splits > 256 || (s + 15) / 16 * splits > 65535)
    return ek_fail(hipErrorInvalidValue, "attn_verify: splits must be 1..256, prompts of 1048560 tokens / splits");
  if (splits > 1 && (!part || part_floats < splits * b * s * n_q * (head_dim + 2)))
    return ek_fail(hipErrorInvalidValue, "attn_verify: the split workspace is too small");
  if (ldq % 8 || ldo % 8 || css % 8 || csh % 8 || csb % 8 || (reinterpret_cast<uintptr_t>(q) & 15) ||
      (reinterpret_cast<uintptr_t>(k_cache) & 15) || (reinterpret_cast<uintptr_t>(v_cache) & 15))
    return ek_fail(hipErrorInvalidValue, "attn_prefill/attn_verify: rows must be 16-byte aligned");
  PrefillParams p;
  memset(&p, 0, sizeof(p));
  p.q = (const bf16_t*)q; p.ldq = ldq;
  p.kc = (const bf16_t*)k_cache; p.vc = (const bf16_t*)v_cache; p.csb = csb; p.csh = csh; p.css = css;
  p.start = start; p.q0 = q0;
  p.out = (bf16_t*)out; p.ldo = ldo;
  p.s = s; p.s_cap = s_cap; p.nkv = (int)n_kv; p.scale = sm_scale;
  p.nq = (int)n_q;
  p.nsplit = (int)splits;
  // keys per split: the cache's rows spread evenly, in whole 32-key tiles
  p.kchunk = ((s_cap + splits - 1) / splits + KB - 1) / KB * KB;
  p.po = part;
  p.pml = part ? part + splits * b * s * n_q * head_dim : nullptr;
  hipStream_t st = (hipStream_t)stream;
  const int g = (int)(n_q / n_kv);
  switch (head_dim) {
    case 32: return launch_prefill_g<32>(p, g, b, st);
    case 64: return launch_prefill_g<64>(p, g, b, st);
    case 128: return launch_prefill_g<128>(p, g, b, st);
    default: return ek_fail(hipErrorInvalidValue, "attn_prefill/attn_verify: head_dim must be 32, 64 or 128");
  }
}

}  // namespace

extern "C" {

int ek_attn_prefill(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, int64_t csb, int64_t csh,
                    int64_t css, int64_t s_cap, const int32_t* start, void* out, int64_t ldo, int64_t b, int64_t s,
                    int64_t n_q, int64_t n_kv, int64_t head_dim, float sm_scale, void* stream) {
  EK_GUARD();
  return attn_flash(q, ldq, k_cache, v_cache, csb, csh, css, s_cap, start, nullptr, out, ldo, b, s, n_q, n_kv,
                    head_dim, sm_scale, stream);
}

int ek_attn_verify(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, int64_t csb, int64_t csh,
                   int64_t css, int64_t s_cap, const int32_t* start, const int64_t* len_b, void* out, int64_t ldo,
                   int64_t b, int64_t nq, int64_t n_q, int64_t n_kv, int64_t head_dim, float sm_scale,
                   float* part, int64_t part_floats, int64_t splits, void* stream) {
  EK_GUARD();
  if (!len_b) return ek_fail(hipErrorInvalidValue, "attn_verify: len_b is required");
  return attn_flash(q, ldq, k_cache, v_cache, csb, csh, css, s_cap, start, len_b, out, ldo, b, nq, n_q, n_kv,
                    head_dim, sm_scale, stream, part, part_floats, splits);
}

}  // extern "C"
