// Device code shared by the convolution kernels: tile mapping, LDS DMA helpers,
// residual loads and epilogues.
#ifndef KGH_CONV_DEVICE_H
#define KGH_CONV_DEVICE_H

#include "kgh_common.h"

#include <climits>
#include <cstdint>
#include <cstdio>
#include <string>
#include <type_traits>

namespace {

template<typename... A>
std::string kernelLabel(const char* fmt, A... a) {
  char buf[160];
  std::snprintf(buf, sizeof(buf), fmt, a...);
  return buf;
}

}  // namespace

namespace {

template<typename T> struct MfmaCfg;

template<> struct MfmaCfg<half_t> {
  static constexpr int BK = 32;      // input channels per K step
  static constexpr int KSUB = 16;    // k per instruction
  static constexpr int LANE_K = 8;   // consecutive k held by one lane
  typedef half8_t Frag;
  __device__ static floatx16 mma(Frag a, Frag b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

constexpr int CONV_BM = 128;
constexpr int CONV_THREADS = 256;
constexpr int CONV_STAGE_LD = 36;  // fp32 row stride of the epilogue's accumulator stage
constexpr int convStageBytes(int WM) { return 4 * (CONV_BM / WM) * CONV_STAGE_LD * 4; }

// Workgroups are dealt round-robin to the 8 XCDs; this remaps blockIdx.x so
// that each XCD owns a contiguous run of row tiles, whose overlapping 3x3
// halo rows then hit in that XCD's L2. A bijection on [0, gridDim.x).
__device__ __forceinline__ int xcdContiguousTile() {
  const int tiles = gridDim.x;
  const int xcd = blockIdx.x & 7;
  const int perXcd = tiles >> 3;
  const int extra = tiles & 7;
  return xcd * perXcd + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3);
}

// Tile coordinates for a 1-D grid of rowTiles x colTiles workgroups: after
// the XCD remap the column tiles of one row tile are consecutive, so they run
// on the same XCD and read the row tile's A operand from that XCD's L2.
__device__ __forceinline__ void rowColTile(int colTiles, int& rowTile, int& colTile) {
  const int id = xcdContiguousTile();
  rowTile = id / colTiles;
  colTile = id - rowTile * colTiles;
}

// Calls f(std::integral_constant<int, ACT>()) for the epilogue's activation
// kind, so the per-element activation is selected at compile time instead of
// branching on every element.
template<typename F>
__host__ __device__ __forceinline__ void withActKind(int act, bool used, F&& f) {
  switch(used ? act : KGH_ACT_IDENTITY) {
    case KGH_ACT_RELU: f(std::integral_constant<int, KGH_ACT_RELU>()); break;
    case KGH_ACT_MISH: f(std::integral_constant<int, KGH_ACT_MISH>()); break;
    case KGH_ACT_SILU: f(std::integral_constant<int, KGH_ACT_SILU>()); break;
    case KGH_ACT_MISH_SCALE8: f(std::integral_constant<int, KGH_ACT_MISH_SCALE8>()); break;
    default: f(std::integral_constant<int, KGH_ACT_IDENTITY>()); break;
  }
}

// Sum of squares of the 16 stored values of this lane, added to its partner
// lane's (the other 16 columns of the same row and 32-column block), stored
// once per block: the producer side of a folded RMSNorm (see ConvEpilogue).
// Both lanes of a pair take this path together (rawEnd is a multiple of 32).
// fp16 values square exactly in fp32; the pairs go through the packed dot
// product (one instruction per two values, no conversions).
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
template<typename T>
__device__ __forceinline__ void storeBlockSumSq(const ConvEpilogue<T>& epi, int m, int c0, const T (&o)[16]) {
  float ss = 0.0f;
  if constexpr(std::is_same<T, half_t>::value) {
#pragma unroll
    for(int j = 0; j < 8; j++) {
      const half2_t h = {o[2 * j], o[2 * j + 1]};
      ss = __builtin_amdgcn_fdot2(h, h, ss, false);
    }
  }
  else {
#pragma unroll
    for(int j = 0; j < 16; j++) {
      const float f = kgh_to_float(o[j]);
      ss += f * f;
    }
  }
  // Partner lane by a DPP quad permutation [1,0,3,2] (no LDS round trip).
  ss += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0xB1, 0xF, 0xF, false));
  if((c0 & 16) == 0) epi.sumSqOut[(size_t)m * epi.ldSq + (c0 >> 5)] = ss;
}

// Loads a wave's RB x CB tiles of a plain residual into the accumulators:
// 16-byte row-major loads (lane: row lane >> 1, channels 16 * (lane & 1)..),
// all issued before the first is used, then a transpose through this wave's
// stage (32 x CONV_STAGE_LD floats) into the matrix-core C layout (lane l,
// register r of tile (rb, cb) is C[(r/4)*8 + (l/32)*4 + r%4][l % 32]). Rows
// at or past M read row M - 1; the epilogue never stores them.
template<typename T, int RB, int CB, int RBATCH = RB>
__device__ __forceinline__ void residualToAcc(floatx16 (&acc)[RB][CB], const T* __restrict__ residual, int ldRes, int mBase,
                                              int nBase, int M, float* stage) {
  constexpr int RV = 16 * (int)sizeof(T) / 16;  // 16-byte vectors per 16 channels
  static_assert(RB % RBATCH == 0, "row blocks are loaded RBATCH at a time");
  const int lane = threadIdx.x & 63;
  const int half = lane & 1;
  const int lrow = lane >> 1;
  const int laneRow = lane & 31;
#pragma unroll
  for(int rb0 = 0; rb0 < RB; rb0 += RBATCH) {
  uint4 raw[RBATCH][CB][RV];
#pragma unroll
  for(int rr = 0; rr < RBATCH; rr++) {
    int m = mBase + (rb0 + rr) * 32 + lrow;
    m = m < M ? m : M - 1;
#pragma unroll
    for(int cb = 0; cb < CB; cb++) {
      const uint4* rp = (const uint4*)(residual + (size_t)m * ldRes + nBase + cb * 32 + half * 16);
#pragma unroll
      for(int q = 0; q < RV; q++) raw[rr][cb][q] = rp[q];
    }
  }
#pragma unroll
  for(int rr = 0; rr < RBATCH; rr++)
#pragma unroll
    for(int cb = 0; cb < CB; cb++) {
      const int rb = rb0 + rr;
      const T* hv = (const T*)raw[rr][cb];
      asm volatile("" ::: "memory");
#pragma unroll
      for(int q = 0; q < 4; q++) {
        float4 f = make_float4(kgh_to_float(hv[4 * q]), kgh_to_float(hv[4 * q + 1]), kgh_to_float(hv[4 * q + 2]),
                               kgh_to_float(hv[4 * q + 3]));
        *(float4*)&stage[lrow * CONV_STAGE_LD + half * 16 + 4 * q] = f;
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for(int r = 0; r < 16; r++) acc[rb][cb][r] = stage[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * CONV_STAGE_LD + laneRow];
    }
  }
  asm volatile("" ::: "memory");
}

typedef __attribute__((address_space(3))) void lds_void_t;

// XOR swizzle of the four 16-byte groups of a 64-byte LDS row. SWZ_SHIFT
// selects which row bits permute the groups: rows that one ds_read_b128 phase
// reads (consecutive rows, same logical group) must land in distinct banks.
// gfx950 serves a 16-lane phase from 64 banks (four 64-byte rows per bank
// line), so the term is (row >> 2) & 3: measured with SQ_LDS_BANK_CONFLICT,
// (row >> 1) & 3 left conflict cycles at ~45% of LDS-active cycles, this
// leaves none in the K loop.
constexpr int SWZ_SHIFT = 2;
__device__ __forceinline__ int swizzleTerm(int row) { return (row >> SWZ_SHIFT) & 3; }
__device__ __forceinline__ int swizzled(int row, int group) { return row * 64 + ((group ^ swizzleTerm(row)) << 4); }
// Physical group of DMA lane l (row 16 j + (l >> 2), slot l & 3) holds
// logical group (l & 3) ^ swizzleTerm(row), independent of j.
__device__ __forceinline__ int dmaLogicalGroup(int lane) { return (lane & 3) ^ swizzleTerm(lane >> 2); }

// s_waitcnt vmcnt(n) (n < 64) leaving the other counters unconstrained: the
// gfx9 encoding keeps vmcnt bits 3:0 in imm[3:0] and bits 5:4 in imm[15:14],
// expcnt in imm[6:4] and lgkmcnt in imm[11:8] (all-ones = no wait).
template<int N>
__device__ __forceinline__ void waitVmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0xF70);
}

// Workgroup barrier without the memory fence of __syncthreads(), whose
// release semantics would wait for every DMA still in flight (vmcnt(0)).
// The empty asm statements keep the compiler from moving memory accesses
// across it; each wave's LDS reads have completed before the barrier (their
// results feed the matrix instructions before it), and the DMA writes a wave
// needs after it are covered by the explicit vmcnt wait before it.
__device__ __forceinline__ void barrierNoFence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Epilogue for one wave's RB x CB block of 32x32 accumulator tiles at rows
// mBase.., columns nBase..; stage is this wave's 32 x CONV_STAGE_LD floats of
// LDS. With RES_IN_ACC the accumulators already hold the residual (loaded
// before the K loop, so its memory latency overlaps the first DMA waits)
// and only the outputs touch memory here. The stage is private to the wave and a wave's LDS operations execute in order, so no
// workgroup barrier is needed; the empty asm statements only keep the
// compiler from reordering the stage accesses.
// nscLds: the folded-RMSNorm row scales of the wave's rows (row r of the
// wave at nscLds[r]) when the kernel computed them, else null (computed here).
template<typename T, int RB, int CB, bool RES_IN_ACC, bool GLU, int ACT, bool ROPE = false>
__device__ __forceinline__ void storeWaveEpilogueAct(floatx16 (&acc)[RB][CB], float* stage, int mBase, int nBase, int M, int HW,
                                                     const ConvEpilogue<T>& epi, const float* nscLds) {
  constexpr int VEC = 16 / (int)sizeof(T);
  constexpr int RV = 16 / VEC;  // 16-byte vectors per lane per block
  const int lane = threadIdx.x & 63;
  const int laneRow = lane & 31;
  const int half = lane & 1;   // which 16-channel half of the 32 columns
  const int lrow = lane >> 1;  // 0..31
  float msk[RB];
  float nsc[RB];  // folded RMSNorm row scales, once per row
  int xyR[RB];    // board positions of the rows (rotary mode)
#pragma unroll
  for(int rb = 0; rb < RB; rb++) {
    const int m = mBase + rb * 32 + lrow;
    msk[rb] = m < M ? epi.mask[m] : 0.0f;
    xyR[rb] = ROPE ? m % HW : 0;
    nsc[rb] = epi.rowNormIn == nullptr || m >= M ? 0.0f : nscLds != nullptr ? nscLds[rb * 32 + lrow] : kgh_row_norm_scale(epi, m, msk[rb]);
  }
#pragma unroll
  for(int cb = 0; cb < CB; cb++) {
    const int c0 = nBase + cb * 32 + half * 16;  // first of this lane's 16 channels
    const bool rawCols = c0 < epi.rawEnd;        // the split points are multiples of 16
    const bool actCols = !ROPE && epi.outAct != nullptr && c0 >= epi.actBegin;
    float aS[16], aB[16];
    if(actCols && !epi.glu) {
#pragma unroll
      for(int j = 0; j < 16; j++) {
        aS[j] = epi.actScale[c0 - epi.actBegin + j];
        aB[j] = epi.actBias[c0 - epi.actBegin + j];
      }
    }
#pragma unroll
    for(int rb = 0; rb < RB; rb++) {
      asm volatile("" ::: "memory");
#pragma unroll
      for(int r = 0; r < 16; r++) stage[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * CONV_STAGE_LD + laneRow] = acc[rb][cb][r];
      asm volatile("" ::: "memory");
      float v[16];
      const float4* src = (const float4*)&stage[lrow * CONV_STAGE_LD + half * 16];
#pragma unroll
      for(int q = 0; q < 4; q++) {
        float4 t = src[q];
        v[4 * q + 0] = t.x;
        v[4 * q + 1] = t.y;
        v[4 * q + 2] = t.z;
        v[4 * q + 3] = t.w;
      }
      const int m = mBase + rb * 32 + lrow;
      if(m < M) {
        if(epi.rowNormIn != nullptr) {
#pragma unroll
          for(int j = 0; j < 16; j++) v[j] *= nsc[rb];
        }
        if(epi.ncBias != nullptr) {
          const float* nb = epi.ncBias + (size_t)(m / HW) * epi.ldNC + c0;
#pragma unroll
          for(int j = 0; j < 16; j++) v[j] += nb[j];
        }
        if(!RES_IN_ACC && epi.residual != nullptr) {
          T rv[16];
          const uint4* rp = (const uint4*)(epi.residual + (size_t)m * epi.ldRes + c0);
#pragma unroll
          for(int q = 0; q < RV; q++) ((uint4*)rv)[q] = rp[q];
#pragma unroll
          for(int j = 0; j < 16; j++) {
            float r = kgh_to_float(rv[j]);
            v[j] = epi.maskResidualAdd ? r + v[j] * msk[rb] : r + v[j];
          }
        }
        if(rawCols) {
          T o[16];
#pragma unroll
          for(int j = 0; j < 16; j++) o[j] = kgh_from_float<T>(v[j]);
          if constexpr(ROPE) {
            if(c0 < epi.ropeEnd) kgh_rope_stored(epi, xyR[rb], HW, c0, o);
          }
          uint4* dst = (uint4*)(epi.outRaw + (size_t)m * epi.ldRaw + c0);
#pragma unroll
          for(int q = 0; q < RV; q++) dst[q] = ((const uint4*)o)[q];
          if(epi.sumSqOut != nullptr) storeBlockSumSq(epi, m, c0, o);
        }
        if constexpr(GLU) {
          if(actCols) {
            T o[8];
#pragma unroll
            for(int j = 0; j < 8; j++) o[j] = kgh_from_float<T>(kgh_activate_fast(v[j], ACT < 0 ? epi.actKind : ACT) * v[8 + j]);
            uint4* dst = (uint4*)(epi.outAct + (size_t)m * epi.ldAct + (c0 - epi.actBegin) / 2);
#pragma unroll
            for(int q = 0; q < RV / 2; q++) dst[q] = ((const uint4*)o)[q];
          }
        }
        else if(actCols) {
          T o[16];
#pragma unroll
          for(int j = 0; j < 16; j++)
            o[j] = kgh_from_float<T>(kgh_activate_fast(v[j] * aS[j] + aB[j], ACT < 0 ? epi.actKind : ACT) * msk[rb]);
          uint4* dst = (uint4*)(epi.outAct + (size_t)m * epi.ldAct + (c0 - epi.actBegin));
#pragma unroll
          for(int q = 0; q < RV; q++) dst[q] = ((const uint4*)o)[q];
        }
      }
    }
  }
}

// ACT_FIXED instantiates the epilogue per activation kind (no per-element
// branch on the kind); kernels with no registers to spare keep one body that
// selects the activation at run time (KGH_ACT_DYNAMIC).
constexpr int KGH_ACT_DYNAMIC = -1;
template<typename T, int RB, int CB, bool RES_IN_ACC, bool GLU, bool ACT_FIXED = true, bool ALLOW_ROPE = false>
__device__ __forceinline__ void storeWaveEpilogue(floatx16 (&acc)[RB][CB], float* stage, int mBase, int nBase, int M, int HW,
                                                  const ConvEpilogue<T>& epi, const float* nscLds = nullptr) {
  if constexpr(ALLOW_ROPE && !GLU) {
    if(epi.ropeEnd > 0) {
      storeWaveEpilogueAct<T, RB, CB, RES_IN_ACC, false, KGH_ACT_IDENTITY, true>(acc, stage, mBase, nBase, M, HW, epi, nscLds);
      return;
    }
  }
  if constexpr(ACT_FIXED) {
    withActKind(epi.actKind, epi.outAct != nullptr, [&](auto actTag) {
      storeWaveEpilogueAct<T, RB, CB, RES_IN_ACC, GLU, decltype(actTag)::value>(acc, stage, mBase, nBase, M, HW, epi, nscLds);
    });
  }
  else {
    storeWaveEpilogueAct<T, RB, CB, RES_IN_ACC, GLU, KGH_ACT_DYNAMIC>(acc, stage, mBase, nBase, M, HW, epi, nscLds);
  }
}

}  // namespace

#endif
