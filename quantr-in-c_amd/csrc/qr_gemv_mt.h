// qr_gemv_mt.h -- row-major Q8_0 / Q6_K GEMV for two to eight tokens on int8
// MFMA: y[t][r] = W[r] . x[t], one weight pass for all tokens.
//
// A workgroup owns tiles of 16 weight rows and cuts their units into stages of
// eight; its waves take the stages in turn.  A stage's bytes come into the
// wave's LDS slot by DMA; per 32-element unit its lanes read them as the B
// operand of v_mfma_i32_16x16x32_i8 (lane -> row lane%16, elements
// 8*(lane/16)..+7) and the tokens' quantized activations as A (lane -> A row
// lane%16, the same elements).  D is lane -> weight row lane%16, A rows
// 4*(lane/16)+i.  The A rows are laid out so that each lane ends with whole
// sums of its own (weight row, token); nothing crosses lanes:
//   sequential order: A row 4g + i is token g + 4i (i = 0, or 0 and 1 for
//     eight tokens), the other A rows zero;
//   Q8_0 lane orders: a unit's eight lane sums are eight A rows of one token,
//     row (token g, lane k) holding only the token's bytes 2k, 2k+1, 16+2k,
//     17+2k (the others zero): A row 4g + i of product j is token g, lane
//     i + 4j, so a lane ends with one token's eight lane accumulators.  Eight
//     tokens are two workgroups of four.
// The integer sums are exact in any order; each fp32 operation is the
// reference's, in its order (term_q8, term_q6, q8_lane_update).  Only the adds
// of the row's running sums are a chain: the waves form their stages' terms
// side by side and hand the sums from stage to stage through LDS.
//
// What bounds it: the latency of a stage (DMA, LDS reads, products, terms: about
// 1.8 us a wave) and the fp32 terms: 5632 x 2048 Q8_0, eight tokens, AVX2 order,
// issues 4.7 M VALU instructions, 7.6 of its 15.7 us, with 2.4 waves per SIMD.  One wave
// doing a tile's whole chain by itself ran at that latency per stage: 5632 x 2048
// Q8_0, eight tokens, AVX2 order 18.9 us against 14.7.  The lane orders' 64 terms
// per lane and stage leave no registers for more than four waves per workgroup
// (8 waves: 17.2 us); the sequential order runs eight (2048 x 5632 Q6_K, four
// tokens: 15.8 us with four, 12.9 with eight; a second slot per wave 13.3).
// Against the kernels that served these calls before, one Q8_0 pass over 5632 x
// 2048: AVX2 order 234.6 -> 14.7 us for eight tokens, 42.9 -> 11.5 for four;
// sequential 20.6 -> 13.3 and 14.7 -> 10.0; Q6_K 2048 x 5632, four tokens,
// 25.9 -> 12.9.
#pragma once

#include <type_traits>

#include "qr_blk.h"
#include "qr_gemv.h"

namespace qr {

constexpr int kMtRows = 16;  // weight rows per tile
constexpr int kMtUnits = 8;  // units per stage

// LDS: the int8 activations [nt][U * 32 + 32] (the 32 bytes of padding put the
// tokens' records of one unit in different banks), then (bd, -32 * bs) pairs
// [nt][U + 1].
__host__ __device__ inline int mt_qstride(int U) { return U * 32 + 32; }
__host__ __device__ inline size_t mt_act_bytes(int U, int nt) {
  return align16((size_t)nt * mt_qstride(U) + (size_t)nt * (U + 1) * 8);
}

// quantize_row_q8_0 (src/quant.c:143-158) of the tokens' first U blocks into
// LDS, four adjacent threads per block; KB batches of loads in flight.  PERM:
// each 8-element group as [x0 x2 x4 x6 | x1 x3 x5 x7].  then() is called once
// the first loads have landed: a DMA issued before them would have to land
// first, one issued after them runs beside the arithmetic.
template <bool PERM, int KB, typename F>
__device__ inline void mt_quantize(const float* __restrict__ x, size_t xstride, int nt, int U,
                                   uint8_t* q, uint2* sc, F then) {
  const int per = 4 * U, total = nt * per, nthr = blockDim.x;
  const int qs = mt_qstride(U);
  for (int base = 0; base < total; base += KB * nthr) {
    float4 f0[KB], f1[KB];
#pragma unroll
    for (int b = 0; b < KB; b++) {
      const int gi = base + b * nthr + (int)threadIdx.x;
      const int t = gi < total ? gi / per : 0, gr = gi < total ? gi - t * per : 0;
      const float4* p = reinterpret_cast<const float4*>(x + t * xstride + (size_t)gr * 8);
      f0[b] = p[0];
      f1[b] = p[1];
    }
    if (base == 0) {
      wait_vmcnt<0>();
      then();
    }
#pragma unroll
    for (int b = 0; b < KB; b++) {
      const int gi = base + b * nthr + (int)threadIdx.x;
      if (base + b * nthr >= total) break;  // uniform
      const float v[8] = {f0[b].x, f0[b].y, f0[b].z, f0[b].w, f1[b].x, f1[b].y, f1[b].z, f1[b].w};
      float amax = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float av = __builtin_fabsf(v[i]);
        amax = av > amax ? av : amax;
      }
      // the block's other groups: the quad's other lanes
      float o = __builtin_bit_cast(
          float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, amax), 0xB1, 0xF, 0xF, false));
      amax = o > amax ? o : amax;
      o = __builtin_bit_cast(
          float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, amax), 0x4E, 0xF, 0xF, false));
      amax = o > amax ? o : amax;
      const float dd = amax / 127.0f;
      const float id = dd != 0.0f ? 1.0f / dd : 0.0f;
      int w[8], s = 0;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        w[i] = (int)(int8_t)(int)__builtin_rintf(v[i] * id);
        s += w[i];
      }
      s += __builtin_amdgcn_update_dpp(0, s, 0xB1, 0xF, 0xF, false);
      s += __builtin_amdgcn_update_dpp(0, s, 0x4E, 0xF, 0xF, false);
      if (gi < total) {
        const int t = gi / per, gr = gi - t * per;
        *reinterpret_cast<uint2*>(q + (size_t)t * qs + (size_t)gr * 8) =
            PERM ? make_uint2(pack4(w[0], w[2], w[4], w[6]), pack4(w[1], w[3], w[5], w[7]))
                 : make_uint2(pack4(w[0], w[1], w[2], w[3]), pack4(w[4], w[5], w[6], w[7]));
        if ((gr & 3) == 0)
          sc[t * (U + 1) + (gr >> 2)] =
              make_uint2(__builtin_bit_cast(uint32_t, qr_h2f(qr_f2h(dd))), (uint32_t)(-32 * s));
      }
    }
  }
}

// A stage of a wave's tile: kMtUnits units of its 16 rows, moved into one of
// the wave's LDS slots by DMA.  A row's stage starts at any even
// address (only its 16-byte chunk does not): kPieces chunks cover it from the
// chunk holding its first byte.
template <int TYPE>
struct MtFmt {
  static constexpr int kBytes = TYPE == QR_T_Q6_K ? QR_Q6K_BYTES : kMtUnits * QR_Q8_BYTES;
  static constexpr int kPieces = (kBytes + 14 + 15) / 16;
  static constexpr int kDma = (kMtRows * kPieces + 63) / 64;  // DMA instructions
  static constexpr int kSlot = kDma * 1024;
};

// A lane's raw bytes of a stage: its 8 elements of each unit and the row's
// scales.
typedef uint64_t mt_u64 __attribute__((aligned(2)));
typedef uint32_t mt_u32 __attribute__((aligned(2)));
template <int TYPE>
struct MtRegs;
template <>
struct MtRegs<QR_T_Q8_0> {
  uint64_t w[kMtUnits];
  uint16_t d[kMtUnits];
};
template <>
struct MtRegs<QR_T_Q6_K> {
  uint32_t ql[kMtUnits];
  uint16_t qh[kMtUnits];
  uint16_t sc[kMtUnits / 2];  // int8 scales of units 2i, 2i + 1
  uint16_t d;
};
__device__ inline void mt_read(const uint8_t* p, int kg, MtRegs<QR_T_Q8_0>& R) {
#pragma unroll
  for (int s = 0; s < kMtUnits; s++) {
    R.w[s] = *reinterpret_cast<const mt_u64*>(p + s * QR_Q8_BYTES + 2 + 8 * kg);
    R.d[s] = *reinterpret_cast<const uint16_t*>(p + s * QR_Q8_BYTES);
  }
}
__device__ inline void mt_read(const uint8_t* p, int kg, MtRegs<QR_T_Q6_K>& R) {
#pragma unroll
  for (int s = 0; s < kMtUnits; s++) {
    R.ql[s] = *reinterpret_cast<const mt_u32*>(p + 16 * s + 4 * kg);
    R.qh[s] = *reinterpret_cast<const uint16_t*>(p + 128 + 8 * s + 2 * kg);
  }
#pragma unroll
  for (int s = 0; s < kMtUnits / 2; s++)
    R.sc[s] = *reinterpret_cast<const uint16_t*>(p + 192 + 2 * s);
  R.d = *reinterpret_cast<const uint16_t*>(p + 208);
}

// Q6_K: a lane's 8 elements q (0..63) of a unit, even elements in the low
// dword: nibbles of ql, bits 4-5 from the 2-bit fields of qh.
__device__ inline uint32_t mt_fields(uint32_t h) {  // 2-bit fields 0, 2, 4, 6 of h -> 4 bytes' bits 4-5
  uint32_t t = h & 0x3333u;
  t = (t | (t << 8)) & 0x00FF00FFu;
  return ((t | (t << 4)) & 0x0F0F0F0Fu) << 4;
}
__device__ inline uint64_t mt_q6(uint32_t ql, uint32_t qh) {
  const uint32_t lo = (ql & 0x0F0F0F0Fu) | mt_fields(qh);
  const uint32_t hi = ((ql >> 4) & 0x0F0F0F0Fu) | mt_fields(qh >> 2);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}

typedef int mt_v4i __attribute__((ext_vector_type(4)));

template <int TYPE, int NT, int Q8O>
struct Mt {
  static constexpr bool kLane = TYPE == QR_T_Q8_0 && Q8O != kQ8Seq;
  static constexpr int kTpl = NT > 4 ? 2 : 1;      // tokens per lane
  static constexpr int kAcc = kLane ? 8 : kTpl;    // chains per lane
  static constexpr int kWaves = kLane ? 4 : 8;     // waves per workgroup
  static constexpr int kRing = kLane ? 2 : 1;      // stages in flight per wave
  static_assert(!kLane || NT <= 4, "a lane order takes four tokens per workgroup");
};
template <int TYPE, int NT, int Q8O>
__host__ __device__ inline size_t mt_lds_bytes(int U) {
  using M = Mt<TYPE, NT, Q8O>;
  // the chains handed over (at most 8 per lane) and the turn
  return mt_act_bytes(U, NT) + (size_t)M::kWaves * M::kRing * MtFmt<TYPE>::kSlot + 64 * 4 * 8 + 16;
}

template <int TYPE, int NT, int Q8O>
__global__ __launch_bounds__((64 * Mt<TYPE, NT, Q8O>::kWaves)) void k_gemv_mt(GemvArgs g) {
  extern __shared__ __align__(16) uint8_t smem[];
  using M = Mt<TYPE, NT, Q8O>;
  using F = MtFmt<TYPE>;
  const int U = qr_units(TYPE, g.d);
  const int lane = threadIdx.x & 63, col = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t rb = qr_wrow_bytes(TYPE, g.d);
  const int ntiles = (g.n + kMtRows - 1) / kMtRows;
  const int nst = (U + kMtUnits - 1) / kMtUnits;  // stages of a tile
  // blockIdx.y: the workgroup's NT tokens
  const float* X = g.X + (size_t)blockIdx.y * NT * g.xstride;
  float* Y = g.Y + (size_t)blockIdx.y * NT * g.ystride;

  uint2* sc = reinterpret_cast<uint2*>(smem + (size_t)NT * mt_qstride(U));
  uint8_t* slots = smem + mt_act_bytes(U, NT) + (size_t)wave * M::kRing * F::kSlot;
  uint8_t* hand = smem + mt_act_bytes(U, NT) + (size_t)M::kWaves * M::kRing * F::kSlot;
  // the sums handed over: a vector of up to four chains per lane, lanes apart
  // by a vector; as LDS pointers, for the order of their accesses holds for LDS
  // instructions only
  typedef float VA __attribute__((ext_vector_type(M::kAcc < 4 ? M::kAcc : 4)));
  constexpr int NV = M::kAcc < 4 ? 1 : M::kAcc / 4;
  typedef __attribute__((address_space(3))) volatile VA LdsVA;
  typedef __attribute__((address_space(3))) volatile int LdsInt;
  LdsVA* hacc = (LdsVA*)(hand) + lane;  // vector i at [64 i]
  LdsInt* turn = (LdsInt*)(hand + 64 * 4 * 8);
  if (threadIdx.x == 0) *turn = 0;

  // DMA: instruction k's lane moves chunk (64 k + lane) % kPieces of row
  // (64 k + lane) / kPieces (past the tile, and past the matrix: the last
  // row); a chunk that is not whole inside the matrix is replaced by the last
  // whole one, and its bytes are stored from registers once the stage has landed
  const size_t total = (size_t)g.n * rb;
  const size_t last = (total & ~(size_t)15) - 16;  // rows are 34 bytes or more
  const int tail = (int)(total & 15);
  // this wave's stages: T = wave, wave + M::kWaves, ... of the workgroup's
  // tiles' stages in order; (it, is) is the next one to issue
  int it = blockIdx.x, is = wave, islot = 0, ahead = 0;
  auto step = [&](int& t, int& s) {
    s += M::kWaves;
    while (s >= nst) {
      s -= nst;
      t += gridDim.x;
    }
  };
  while (is >= nst) {
    is -= nst;
    it += gridDim.x;
  }
  int tile = it, st = is;
  auto issue = [&]() {
    if (it >= ntiles) return;
    const uint32_t dst = lds_u32addr(slots + islot * F::kSlot);
#pragma unroll
    for (int k = 0; k < F::kDma; k++) {
      const int c = k * 64 + lane;
      const int r = min(it * kMtRows + min(c / F::kPieces, kMtRows - 1), g.n - 1);
      size_t o = (((size_t)r * rb + (size_t)(is * F::kBytes)) & ~(size_t)15) + 16 * (c % F::kPieces);
      o = o < last ? o : last;
      lds_dma16_nt(g.W + o, dst + (uint32_t)(k * 1024));
    }
    islot = islot + 1 == M::kRing ? 0 : islot + 1;
    ahead++;
    step(it, is);
  };
  mt_quantize<TYPE == QR_T_Q6_K, 4>(X, (size_t)g.xstride, NT, U, smem, sc, [&]() {
#pragma unroll
    for (int k = 0; k < M::kRing; k++) issue();
  });
  __syncthreads();

  // A operand: row m = lane % 16 (see above); rows without a token read
  // token 0 under a zero mask
  int at;
  bool on;
  uint64_t m0, m1 = 0;
  if constexpr (M::kLane) {
    at = col >> 2;
    on = at < NT;
    const uint64_t m = 0xFFFFull << (16 * (col & 3));
    m0 = on && (kg & 1) == 0 ? m : 0;
    m1 = on && (kg & 1) == 1 ? m : 0;
  } else {
    at = (col >> 2) + 4 * (col & 3);
    on = (col & 3) < M::kTpl && at < NT;
    m0 = on ? ~0ull : 0;
  }
  const uint8_t* ap = smem + (size_t)(on ? at : 0) * mt_qstride(U) + 8 * kg;
  // D: this lane's tokens
  const uint2* sp[M::kTpl];
#pragma unroll
  for (int i = 0; i < M::kTpl; i++) {
    const int t = kg + 4 * i;
    sp[i] = sc + (size_t)(t < NT ? t : 0) * (U + 1);
  }

  int slot = 0;
  for (int T = wave; tile < ntiles; T += M::kWaves, step(tile, st)) {
    // this stage has landed when only the later ones' loads are in flight
    // (stores of outputs, also counted, only make the wait longer)
    if (M::kRing > 1 && ahead > 1) wait_vmcnt<F::kDma*(M::kRing - 1)>();
    else wait_vmcnt<0>();
    ahead--;
    uint8_t* sp0 = slots + slot * F::kSlot;
    slot = slot + 1 == M::kRing ? 0 : slot + 1;
    if (tail && st == nst - 1 && tile == ntiles - 1) {
      const size_t row0 = (size_t)(g.n - 1) * rb + (size_t)st * F::kBytes;
      uint8_t* dst = sp0 + (g.n - 1 - tile * kMtRows) * (16 * F::kPieces) +
                     ((total & ~(size_t)15) - (row0 & ~(size_t)15));
      if (2 * lane < tail)
        *reinterpret_cast<uint16_t*>(dst + 2 * lane) =
            *reinterpret_cast<const uint16_t*>(g.W + (total - tail) + 2 * lane);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    const uint32_t mrow = (uint32_t)min(tile * kMtRows + col, g.n - 1) * (uint32_t)rb;
    MtRegs<TYPE> L;
    mt_read(sp0 + col * (16 * F::kPieces) + ((mrow + (uint32_t)(st * F::kBytes)) & 15u), kg, L);
    const int u0 = st * kMtUnits, cnt = min(kMtUnits, U - u0);
    // the stage's activations (units past the row's last: its last one's)
    uint64_t x[kMtUnits];
    uint2 sv[kMtUnits][M::kTpl];
#pragma unroll
    for (int s = 0; s < kMtUnits; s++) {
      const int u = TYPE == QR_T_Q6_K ? u0 + s : min(u0 + s, U - 1);
      x[s] = *reinterpret_cast<const uint64_t*>(ap + 32 * u);
#pragma unroll
      for (int i = 0; i < M::kTpl; i++) sv[s][i] = sp[i][u];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot is free again
    issue();

    // the products, and the terms without their chain: P[s][k]
    float P[kMtUnits][M::kAcc];
    float dq = 0.0f;
    if constexpr (TYPE == QR_T_Q6_K) dq = qr_h2f(L.d);
#pragma unroll
    for (int s = 0; s < kMtUnits; s++) {
      if constexpr (M::kLane) {
        const mt_v4i z = {0, 0, 0, 0};
        const mt_v4i D0 =
            __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(x[s] & m0), (long)L.w[s], z, 0, 0, 0);
        const mt_v4i D1 =
            __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(x[s] & m1), (long)L.w[s], z, 0, 0, 0);
        const float dd = qr_h2f(L.d[s]) * __builtin_bit_cast(float, sv[s][0].x);
#pragma unroll
        for (int k = 0; k < 4; k++) {
          P[s][k] = (float)D0[k];
          P[s][4 + k] = (float)D1[k];
        }
        if constexpr (Q8O == kQ8Avx512) {
          sv[s][0].x = __builtin_bit_cast(uint32_t, dd);  // joined in the chain's fused step
        } else {
#pragma unroll
          for (int k = 0; k < 8; k++) P[s][k] *= dd;
        }
      } else {
        mt_v4i c = {0, 0, 0, 0};
        if constexpr (TYPE == QR_T_Q6_K) {
#pragma unroll
          for (int i = 0; i < M::kTpl; i++) c[i] = (int)sv[s][i].y;
        }
        uint64_t w;
        if constexpr (TYPE == QR_T_Q6_K) w = mt_q6(L.ql[s], L.qh[s]);
        else w = L.w[s];
        const mt_v4i D =
            __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(x[s] & m0), (long)w, c, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < M::kTpl; i++) {
          const float bd = __builtin_bit_cast(float, sv[s][i].x);
          if constexpr (TYPE == QR_T_Q6_K)  // term_q6
            P[s][i] = ((float)(int8_t)(L.sc[s >> 1] >> (8 * (s & 1))) * dq) * (float)D[i] * bd;
          else  // term_q8
            P[s][i] = (float)D[i] * qr_h2f(L.d[s]) * bd;
        }
      }
    }

    // the chains, in stage order: take them over from the wave of stage T - 1
    // (turn counts the finished stages; a wave's LDS reads are served in order,
    // so sums read after a turn of T are that wave's), add this stage's terms
    // and hand them on.  Every stage before T is some wave's current or earlier
    // one, and the wave of the earliest unfinished one waits for nobody.
#pragma unroll
    for (int s = 0; s < kMtUnits; s++)
#pragma unroll
      for (int k = 0; k < M::kAcc; k++)
        asm volatile("" : "+v"(P[s][k]));  // formed before the wait, not sunk below it
    VA hv[NV];
    for (;;) {
      const int t = __builtin_amdgcn_readfirstlane(*turn);
#pragma unroll
      for (int i = 0; i < NV; i++) hv[i] = hacc[64 * i];
      if (t == T) break;
    }
    float acc[M::kAcc];
#pragma unroll
    for (int k = 0; k < M::kAcc; k++) {
      if constexpr (M::kAcc == 1) acc[k] = hv[0].x;
      else acc[k] = hv[k >> 2][k & 3];
    }
    if (st == 0) {
#pragma unroll
      for (int k = 0; k < M::kAcc; k++) acc[k] = 0.0f;
    }
#pragma unroll
    for (int s = 0; s < kMtUnits; s++) {
      if (TYPE == QR_T_Q6_K || s < cnt) {
#pragma unroll
        for (int k = 0; k < M::kAcc; k++) {
          if constexpr (M::kLane && Q8O == kQ8Avx512)
            acc[k] = q8_lane_update<Q8O>(P[s][k], __builtin_bit_cast(float, sv[s][0].x), acc[k]);
          else
            acc[k] = P[s][k] + acc[k];
        }
      }
    }
    if (st != nst - 1) {
#pragma unroll
      for (int i = 0; i < NV; i++) {
        VA v;
        if constexpr (M::kAcc == 1) {
          v.x = acc[0];
        } else {
#pragma unroll
          for (int k = 0; k < (M::kAcc < 4 ? M::kAcc : 4); k++) v[k] = acc[4 * i + k];
        }
        hacc[64 * i] = v;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    *turn = T + 1;
    if (st == nst - 1) {
      const int row = tile * kMtRows + col;
#pragma unroll
      for (int i = 0; i < M::kTpl; i++) {
        const int t = kg + 4 * i;
        float v = acc[i];
        if constexpr (M::kLane) {
          v = 0.0f;
#pragma unroll
          for (int k = 0; k < 8; k++) v += acc[k];
        }
        if (row < g.n && t < NT) Y[(size_t)t * g.ystride + row] = v;
      }
    }
  }
}

}  // namespace qr
