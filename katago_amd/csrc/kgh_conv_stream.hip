// fp16 convolutions with streamed weights (convStreamKernel) and their weight
// layout.
#include "kgh_conv_device.h"
#include "kgh_conv_stream.h"

#include <utility>

namespace {

// ---------------------------------------------------------------------------
// fp16 1x1 and 3x3 convolution with streamed weights, any board size. A
// workgroup's input rows (its output rows and, for 3x3, one board row and one
// position either side) are DMA'd into LDS once with all their channels; the
// weights never touch LDS: each wave reads its fragments from a second
// prepared layout (prepareFragWeightsKernel) in which a fragment load of a
// wave is one contiguous 1 KB run, through a ring of DEPTH steps of
// registers. One barrier per launch; after it every wave runs its chain of K
// steps (chunk outer, tap inner: the order of every other kernel, so the rows
// are bitwise theirs) with nothing to wait for but its own loads.
//
// What bounds it: with one workgroup per CU (few boards) a wave's chain, 18
// matrix instructions of 36 to 48 cycles per chunk and 32 x 32 block; with
// every CU full the matrix cores (96 boards of 192 channels: 35.5 us, 0.65
// PFLOP/s of the 1.16 a large product reaches). The kernels it replaces loaded
// weights through LDS with a barrier per tap; 192 -> 192 channels, us per
// launch by what forwards gained: one board 14.4 -> 6.4, 16 boards 15.4 ->
// 10.1, 24 boards of 9x9 33.8 -> 7.2, 96 boards of 13x13 46 -> 20.
//
// LDS rows hold cinPad channels and a 16-byte gap: 16 consecutive rows of a
// ds_read_b128 phase start 4 (mod 64) banks times an odd number apart, so
// they fall in distinct bank groups. A tap that leaves the board reads a row
// of zeros: the nine addresses per row block are computed once, and the K loop
// has no masking.
constexpr int STREAM_STAGE_BYTES = 32 * CONV_STAGE_LD * 4;  // a wave's epilogue stage
constexpr int STREAM_RES_BYTES = 16 * CONV_STAGE_LD * 4;    // a wave's residual stage

template<int KS, int BM, int NW>
__host__ __device__ constexpr int streamFixedBytes() {
  return NW * STREAM_RES_BYTES + (KS == 1 ? BM * 4 : 0);
}

// Bytes of dynamic LDS: the row scales, the window (whole 1 KB wave-loads) and
// the row of zeros. The window becomes the waves' epilogue stages.
template<int KS, int BM, int NW>
__host__ __device__ inline int streamLdsBytes(int cinPad, int W) {
  const int rows = BM + (KS == 3 ? 2 * (W + 1) : 0);
  const int strideB = cinPad * 2 + 16;
  const int win = (rows * strideB + 1023) / 1024 * 1024 + (KS == 3 ? strideB : 0);
  return streamFixedBytes<KS, BM, NW>() + (win > NW * STREAM_STAGE_BYTES ? win : NW * STREAM_STAGE_BYTES);
}

// Division by multiplication: divBy(v, divMagic(d)) is v / d for every v with
// 4 v d < 2^32 (the host checks the ranges; doubling both sides gives d = 1 a
// 32-bit factor too).
__device__ __forceinline__ unsigned divBy(unsigned v, unsigned magic) { return __umulhi(v << 1, magic); }

// Seven words fill the gap before the epilogue in the kernel's arguments: with
// one argument more the grid size behind them falls into another 64-byte line,
// and a launch at one board takes 6.85 us instead of 6.66.
struct StreamDims {
  unsigned per, perMagic;  // 16-byte slots per window row
  unsigned hwMagic, wMagic, colTiles, colMagic;
  unsigned partChunks;  // PARTS: chunks per sum
};

// The plain form of the epilogue (raw and activated outputs, per-board bias):
// four lanes take the 64 bytes of a row's 32-column block, so every store
// instruction writes whole 64-byte runs. ADD_RES adds a residual that the lane
// holds in the same places.
template<int RB, int CB, int ACT, bool ADD_RES>
__device__ __forceinline__ void storeWaveRows(floatx16 (&acc)[RB][CB], float* stage, int mBase, int nBase, int M, int HW,
                                              const ConvEpilogue<half_t>& epi, const half8_t (&res)[RB][CB][2]) {
  const int lane = threadIdx.x & 63;
  const int laneRow = lane & 31;
  const int q = lane & 3;       // which 8 of the 32 columns
  const int lrow = lane >> 2;   // 0..15
  float msk[RB][2];
#pragma unroll
  for(int rb = 0; rb < RB; rb++)
#pragma unroll
    for(int p = 0; p < 2; p++) msk[rb][p] = epi.mask[min(mBase + rb * 32 + p * 16 + lrow, M - 1)];
#pragma unroll
  for(int cb = 0; cb < CB; cb++) {
    const int c0 = nBase + cb * 32 + q * 8;
    const bool rawCols = c0 < epi.rawEnd;
    const bool actCols = epi.outAct != nullptr && c0 >= epi.actBegin;
    float aS[8], aB[8];
    if(actCols) {
#pragma unroll
      for(int j = 0; j < 8; j++) {
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
      float v[2][8];
#pragma unroll
      for(int p = 0; p < 2; p++)
#pragma unroll
        for(int h = 0; h < 2; h++) {
          const float4 t = *(const float4*)&stage[(p * 16 + lrow) * CONV_STAGE_LD + q * 8 + h * 4];
          v[p][4 * h] = t.x;
          v[p][4 * h + 1] = t.y;
          v[p][4 * h + 2] = t.z;
          v[p][4 * h + 3] = t.w;
        }
#pragma unroll
      for(int p = 0; p < 2; p++) {
        const int m = mBase + rb * 32 + p * 16 + lrow;
        if(m < M) {
          if(epi.ncBias != nullptr) {
            const float* nb = epi.ncBias + (size_t)(m / HW) * epi.ldNC + c0;
#pragma unroll
            for(int j = 0; j < 8; j++) v[p][j] += nb[j];
          }
          if(ADD_RES && epi.residual != nullptr) {
#pragma unroll
            for(int j = 0; j < 8; j++) v[p][j] = (float)res[rb][cb][p][j] + v[p][j];
          }
          if(rawCols) {
            half8_t o;
#pragma unroll
            for(int j = 0; j < 8; j++) o[j] = (half_t)v[p][j];
            *(half8_t*)(epi.outRaw + (size_t)m * epi.ldRaw + c0) = o;
          }
          if(actCols) {
            half8_t o;
#pragma unroll
            for(int j = 0; j < 8; j++) o[j] = (half_t)(kgh_activate_fast(v[p][j] * aS[j] + aB[j], ACT < 0 ? epi.actKind : ACT) * msk[rb][p]);
            *(half8_t*)(epi.outAct + (size_t)m * epi.ldAct + (c0 - epi.actBegin)) = o;
          }
        }
      }
    }
  }
}

// PARTS (3x3, low-latency mode): every partChunks 32-channel chunks have a sum
// of their own, started at zero; the sums are added in order, then the bias
// and the residual. Additions after each part wait for the matrix core: 0.7 us
// of 7.4 at 192 channels and one board (b18c384nbt's forward 812 us, 762 with
// one sum); a second set of accumulators, added and cleared during the next
// part's instructions, was slower (861 us where this form took 836).
template<int KS, int RB, int CB, int WM, int WN, int DEPTH, bool GLU, bool PARTS>
__global__ __launch_bounds__(64 * WM * WN, 1) void convStreamKernel(const half_t* __restrict__ x, int cinStride, int cinPad, int cout,
                                                                    const half_t* __restrict__ wf, BoardGeom g, StreamDims sd,
                                                                    ConvEpilogue<half_t> epi) {
  constexpr int NW = WM * WN;
  constexpr int NT = 64 * NW;
  constexpr int BM = 32 * RB * WM;
  constexpr int BN = 32 * CB * WN;
  constexpr int TAPS = KS * KS;
  static_assert(KS == 1 || 9 % DEPTH == 0, "a ring slot per tap");
  extern __shared__ __attribute__((aligned(1024))) unsigned char streamLds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM;
  const int wn = wave / WM;
  const int laneRow = lane & 31;
  const int kq = lane >> 5;
  const int HW = g.H * g.W;
  const int M = g.batch * HW;
  const unsigned tile = xcdContiguousTile();
  const unsigned rowTile = divBy(tile, sd.colMagic);
  const int m0 = rowTile * BM;
  const int n0 = (tile - rowTile * sd.colTiles) * BN;
  const int halo = KS == 3 ? g.W + 1 : 0;
  const int winRows = BM + 2 * halo;
  const int strideB = cinPad * 2 + 16;
  const int chunks = cinPad / 32;
  const int mWave = m0 + wm * 32 * RB;
  const int nWave = n0 + wn * 32 * CB;
  float* resStage = (float*)(streamLds + wave * STREAM_RES_BYTES);
  float* rowScale = (float*)(streamLds + NW * STREAM_RES_BYTES);
  unsigned char* win = streamLds + streamFixedBytes<KS, BM, NW>();
  float* stage = (float*)(win + wave * STREAM_STAGE_BYTES);
  const int winBytes = (winRows * strideB + 1023) / 1024 * 1024;

  // The residual starts the accumulators (or waits for the end), so its loads
  // come first: four lanes per 64-byte row of a 32 x 32 block.
  const bool loadRes = epi.residual != nullptr && !epi.maskResidualAdd;
  const bool resInAcc = !PARTS && loadRes;
  const int quarter = lane & 3, qRow = lane >> 2;
  half8_t res[RB][CB][2];
  if(loadRes) {
#pragma unroll
    for(int rb = 0; rb < RB; rb++)
#pragma unroll
      for(int p = 0; p < 2; p++) {
        const half_t* src = epi.residual + (size_t)min(mWave + rb * 32 + p * 16 + qRow, M - 1) * epi.ldRes + nWave + quarter * 8;
#pragma unroll
        for(int cb = 0; cb < CB; cb++) res[rb][cb][p] = *(const half8_t*)(src + cb * 32);
      }
  }

  // Window slot q (16 bytes) is group q % per of window row q / per, the last
  // group being the gap; wave-load j fills slots 64 j .. 64 j + 63. Rows
  // outside [0, M) only feed taps that read zeros, or outputs that are never
  // stored; the slots past the last row and the gaps load a valid address.
  // Byte offsets are 32-bit: the host keeps tensors below 2^31 elements.
  const int loads = winBytes / 1024;
  for(int j = wave; j < loads; j += NW) {
    const unsigned slot = j * 64 + lane;
    const unsigned row = divBy(slot, sd.perMagic);
    const unsigned grp = min(slot - row * sd.per, sd.per - 2);
    const int gm = min(max(m0 - halo + (int)row, 0), M - 1);
    const unsigned off = ((unsigned)gm * (unsigned)cinStride + grp * 8) * 2;
    __builtin_amdgcn_global_load_lds((const void*)((const char*)x + off), (lds_void_t*)(win + j * 1024), 16, 0, 0);
  }
  if constexpr(KS == 3) {
    for(int i = tid * 16; i < strideB; i += NT * 16) *(uint4*)(win + winBytes + i) = make_uint4(0, 0, 0, 0);
  }

  // Weight fragments of step s = chunk * TAPS + tap: 2 CB runs of 1 KB.
  const int steps = chunks * TAPS;
  const int nBlocks = cout / 32;
  const unsigned laneOff = lane * 16;
  half8_t bRing[DEPTH][CB][2];
  auto loadB = [&](int s, half8_t (&b)[CB][2]) {
    const char* p = (const char*)wf + ((size_t)s * nBlocks + nWave / 32) * 2048;
#pragma unroll
    for(int cb = 0; cb < CB; cb++)
#pragma unroll
      for(int ks = 0; ks < 2; ks++) b[cb][ks] = *(const half8_t*)(p + laneOff + cb * 2048 + ks * 1024);
  };
#pragma unroll
  for(int d = 0; d < DEPTH; d++) loadB(KS == 3 ? d : min(d, steps - 1), bRing[d]);

  // The epilogue's operands into this XCD's L2 while the window loads: one
  // access per 4 bytes of the wave's mask rows and activation parameters.
  float touched = epi.mask[min(mWave + (RB == 1 ? laneRow : lane), M - 1)];
  if(epi.outAct != nullptr && !epi.glu && nWave + laneRow >= epi.actBegin)
    touched += (kq ? epi.actBias : epi.actScale)[nWave + laneRow - epi.actBegin];
  const bool rowNorm = KS == 1 && epi.rowNormIn != nullptr;
  if constexpr(KS == 1) {
    if(rowNorm) {
      for(int i = tid; i < BM; i += NT) {
        float nq[KGH_NORM_MAX_BLOCKS], nMask = 0.0f;
        const bool live = m0 + i < M;
        if(live) kgh_row_norm_load(epi, m0 + i, nq, nMask);
        rowScale[i] = live ? kgh_row_norm_finish(epi, nq, nMask) : 0.0f;
      }
    }
  }

  // LDS byte address of the lane's A fragments per tap (channel 0 of its k
  // group).
  int aAddr[RB][TAPS];
#pragma unroll
  for(int rb = 0; rb < RB; rb++) {
    const int r = wm * 32 * RB + rb * 32 + laneRow;
    if constexpr(KS == 3) {
      const int m = m0 + r;
      const int sp = m - (int)divBy(m, sd.hwMagic) * HW;
      const int y = divBy(sp, sd.wMagic);
      const int xx = sp - y * g.W;
      const bool yOk[3] = {m < M && y > 0, m < M, m < M && y < g.H - 1};
      const bool xOk[3] = {xx > 0, true, xx < g.W - 1};
      const int base = (r + halo) * strideB + kq * 16;
#pragma unroll
      for(int t = 0; t < 9; t++) {
        // A tap that leaves the board reads the row of zeros.
        aAddr[rb][t] = yOk[t / 3] && xOk[t % 3] ? base + ((t / 3 - 1) * g.W + (t % 3 - 1)) * strideB : winBytes + kq * 16;
      }
    }
    else {
      aAddr[rb][0] = r * strideB + kq * 16;
    }
  }
  floatx16 acc[RB][CB];
  if(resInAcc) {
    // Into the matrix-core C layout, 16 rows at a time through a small stage
    // of the wave's own (the window is still loading).
#pragma unroll
    for(int rb = 0; rb < RB; rb++)
#pragma unroll
      for(int cb = 0; cb < CB; cb++)
#pragma unroll
        for(int p = 0; p < 2; p++) {
          asm volatile("" ::: "memory");
#pragma unroll
          for(int h = 0; h < 2; h++) {
            floatx4 f;
#pragma unroll
            for(int j = 0; j < 4; j++) f[j] = (float)res[rb][cb][p][4 * h + j];
            *(floatx4*)&resStage[qRow * CONV_STAGE_LD + quarter * 8 + h * 4] = f;
          }
          asm volatile("" ::: "memory");
#pragma unroll
          for(int k = 0; k < 8; k++) acc[rb][cb][p * 8 + k] = resStage[((k >> 2) * 8 + kq * 4 + (k & 3)) * CONV_STAGE_LD + laneRow];
        }
    asm volatile("" ::: "memory");
  }
  else {
#pragma unroll
    for(int rb = 0; rb < RB; rb++)
#pragma unroll
      for(int cb = 0; cb < CB; cb++)
#pragma unroll
        for(int r = 0; r < 16; r++) acc[rb][cb][r] = 0.0f;
  }
  asm volatile("" ::"v"(touched));
  waitVmcnt<0>();
  __syncthreads();

  auto readA = [&](int tap, int c, int rb, int ks) { return *(const half8_t*)(win + aAddr[rb][tap] + c * 64 + ks * 32); };
  auto readB = [&](int s, int cb, int ks) {
    return *(const half8_t*)((const char*)wf + ((size_t)s * nBlocks + nWave / 32) * 2048 + laneOff + cb * 2048 + ks * 1024);
  };
  // One K step: its matrix instructions on a and b, with the fragment reads
  // of a later step (nextA into an, nextB over b once its half is used) one
  // after each instruction, so that they issue while the matrix core works.
  // Left to itself the compiler moves every load down to its use.
  auto step = [&](half8_t (&a)[RB][2], half8_t (&b)[CB][2], half8_t (&an)[RB][2], auto&& nextA, auto&& nextB) {
#pragma unroll
    for(int i = 0; i < 2 * RB * CB; i++) {
      const int ks = i / (RB * CB), rb = i / CB % RB, cb = i % CB;
      // One tile per wave is one chain of dependent instructions: its reads
      // come ahead of them.
      if(RB * CB == 1 && i == 0) {
        nextA(an[0][0], 0, 0);
        nextA(an[0][1], 0, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[rb][ks], b[cb][ks], acc[rb][cb], 0, 0, 0);
      if(RB * CB > 1 && i < 2 * RB) nextA(an[i >> 1][i & 1], i >> 1, i & 1);
      if(rb == RB - 1) nextB(b[cb][ks], cb, ks);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr(KS == 3) {
    // Three A slots, read two steps ahead (9 % 3 == 0).
    half8_t aRing[3][RB][2];
#pragma unroll
    for(int t = 0; t < 2; t++)
#pragma unroll
      for(int rb = 0; rb < RB; rb++)
#pragma unroll
        for(int ks = 0; ks < 2; ks++) aRing[t][rb][ks] = readA(t, 0, rb, ks);
    auto chunk = [&](int c, auto lastTag) {
      constexpr bool LAST = decltype(lastTag)::value;
#pragma unroll
      for(int t = 0; t < 9; t++) {
        step(
          aRing[t % 3], bRing[t % DEPTH], aRing[(t + 2) % 3],
          [&](half8_t& f, int rb, int ks) {
            if(t < 7) f = readA(t + 2, c, rb, ks);
            else if(!LAST) f = readA(t - 7, c + 1, rb, ks);
          },
          [&](half8_t& f, int cb, int ks) {
            if(!LAST || t + DEPTH < 9) f = readB(9 * c + t + DEPTH, cb, ks);
          });
      }
    };
    if constexpr(PARTS) {
      static_assert(RB == 1 && CB == 1, "registers for the sum");
      floatx16 sum = acc[0][0];
      unsigned left = sd.partChunks;
      for(int c = 0; c + 1 < chunks; c++) {
        chunk(c, std::integral_constant<bool, false>());
        if(--left == 0) {
          left = sd.partChunks;
#pragma unroll
          for(int r = 0; r < 16; r++) {
            sum[r] += acc[0][0][r];
            acc[0][0][r] = 0.0f;
          }
        }
      }
      chunk(chunks - 1, std::integral_constant<bool, true>());
      acc[0][0] = sum + acc[0][0];
    }
    else {
      for(int c = 0; c + 1 < chunks; c++) chunk(c, std::integral_constant<bool, false>());
      chunk(chunks - 1, std::integral_constant<bool, true>());
    }
  }
  else {
    // Two A slots, read one step ahead; reads past the last step repeat it.
    half8_t aRing[2][RB][2];
    static_assert(DEPTH % 2 == 0, "two A slots");
#pragma unroll
    for(int rb = 0; rb < RB; rb++)
#pragma unroll
      for(int ks = 0; ks < 2; ks++) aRing[0][rb][ks] = readA(0, 0, rb, ks);
    int i = 0;
    for(; i + DEPTH < steps; i += DEPTH) {
#pragma unroll
      for(int d = 0; d < DEPTH; d++)
        step(
          aRing[d & 1], bRing[d], aRing[(d + 1) & 1], [&](half8_t& f, int rb, int ks) { f = readA(0, i + d + 1, rb, ks); },
          [&](half8_t& f, int cb, int ks) { f = readB(min(i + d + DEPTH, steps - 1), cb, ks); });
    }
#pragma unroll
    for(int d = 0; d < DEPTH; d++) {
      if(i + d < steps)
        step(
          aRing[d & 1], bRing[d], aRing[(d + 1) & 1], [&](half8_t& f, int rb, int ks) { f = readA(0, min(i + d + 1, steps - 1), rb, ks); },
          [&](half8_t&, int, int) {});
    }
  }

  __syncthreads();  // every wave is done with the window before it holds the stages
  if constexpr(!GLU) {
    if(epi.sumSqOut == nullptr && !rowNorm && epi.ropeEnd == 0 && (loadRes || epi.residual == nullptr)) {
      withActKind(epi.actKind, epi.outAct != nullptr, [&](auto actTag) {
        storeWaveRows<RB, CB, decltype(actTag)::value, PARTS>(acc, stage, mWave, nWave, M, HW, epi, res);
      });
      return;
    }
  }
  ConvEpilogue<half_t> e = epi;
  if(resInAcc) e.residual = nullptr;
  storeWaveEpilogue<half_t, RB, CB, false, GLU, KS == 1, KS == 1>(acc, stage, mWave, nWave, M, HW, e, rowNorm ? rowScale + wm * 32 * RB : nullptr);
}

// The streamed kernel's weight layout: for each (32-channel chunk, tap,
// 32-column block, 16-channel half) 64 lanes x 8 channels, lane l = column
// l % 32, channels 8 (l / 32) .. + 7 of the half: a wave's fragment is one
// contiguous 1 KB run.
__global__ void prepareFragWeightsKernel(const float* __restrict__ src, half_t* __restrict__ dst, int cout, int cin, int cinPad, int ks) {
  const int taps = ks * ks;
  const long total = (long)taps * cout * cinPad;
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if(idx >= total) return;
  const int lane = (int)(idx >> 3) & 63;
  const long blk = idx >> 10;
  const int nb = (int)(blk % (cout / 32));
  const long step = blk / (cout / 32);
  const int tap = (int)(step % taps);
  const int oc = nb * 32 + (lane & 31);
  const int ic = (int)(step / taps) * 32 + ((int)(idx >> 9) & 1) * 16 + (lane >> 5) * 8 + (int)(idx & 7);
  dst[idx] = ic < cin ? (half_t)src[(((size_t)oc * cin + ic) * ks + tap / ks) * ks + tap % ks] : (half_t)0.0f;
}

constexpr int STREAM_MAX_LDS = 160 * 1024;

inline unsigned divMagic(unsigned d) { return (unsigned)((0x100000000ull + 2ull * d - 1) / (2ull * d)); }

template<int KS, int RB, int CB, int WM, int WN, int DEPTH>
struct Stream {
  static constexpr int BM = 32 * RB * WM, BN = 32 * CB * WN, NW = WM * WN;
  static bool fits(int cinStride, int cinPad, int cout, BoardGeom g, const ConvEpilogue<half_t>& epi) {
    const long HW = (long)g.H * g.W, M = g.batch * HW;
    const long slots = (long)STREAM_MAX_LDS / 16;
    return cinPad % 32 == 0 && cinStride % 8 == 0 && cout % BN == 0 && M * cinStride < (1L << 31) &&
           (long)KS * KS * cout * cinPad < (1L << 31) && (KS == 1 || (!epi.maskResidualAdd && !epi.glu && epi.rowNormIn == nullptr && epi.ropeEnd == 0)) &&
           // the exact ranges of the divisions by multiplication
           4 * (M + BM) * HW < (1L << 32) && 4 * slots * (cinPad / 8 + 1) < (1L << 32) &&
           4 * ((M + BM) / BM * (cout / BN)) * (cout / BN) < (1L << 32) &&
           streamLdsBytes<KS, BM, NW>(cinPad, g.W) <= STREAM_MAX_LDS;
  }
  template<bool GLU, bool PARTS>
  static void run(const half_t* x, int cinStride, int cinPad, int cout, const half_t* wf, BoardGeom g, const ConvEpilogue<half_t>& epi,
                  int partChunks, hipStream_t stream) {
    const int M = g.batch * g.H * g.W;
    const int colTiles = cout / BN;
    const dim3 grid((M + BM - 1) / BM * colTiles), block(64 * NW);
    const int lds = streamLdsBytes<KS, BM, NW>(cinPad, g.W);
    const unsigned per = cinPad / 8 + 1;
    const StreamDims sd = {per, divMagic(per), divMagic(g.H * g.W), divMagic(g.W), (unsigned)colTiles, divMagic(colTiles),
                           (unsigned)partChunks};
    hipLaunchKernelGGL((convStreamKernel<KS, RB, CB, WM, WN, DEPTH, GLU, PARTS>), grid, block, lds, stream, x, cinStride, cinPad, cout,
                       wf, g, sd, epi);
    KGH_CHECK_LAUNCH();
  }
  // w: the prepared weights; the fragment layout follows the first.
  static void launch(const half_t* x, int cinStride, int cinPad, int cout, const half_t* w, BoardGeom g, const ConvEpilogue<half_t>& epi,
                     hipStream_t stream) {
    static const std::string name = kernelLabel("convStreamKernel<%dx%d fp16, %dx%d tiles, %d waves of %dx%d>", KS, KS, BM, BN, NW,
                                                32 * RB, 32 * CB);
    kgh::g_lastConvKernel = name.c_str();
    const half_t* wf = w + (size_t)KS * KS * cout * cinPad;
    if constexpr(KS == 1) {
      if(epi.glu) {
        run<true, false>(x, cinStride, cinPad, cout, wf, g, epi, 0, stream);
        return;
      }
    }
    run<false, false>(x, cinStride, cinPad, cout, wf, g, epi, 0, stream);
  }
  static void launchParts(const half_t* x, int cinStride, int cinPad, int cout, const half_t* w, BoardGeom g,
                          const ConvEpilogue<half_t>& epi, int partChunks, hipStream_t stream) {
    static const std::string name = kernelLabel("convStreamKernel<%dx%d fp16, %dx%d tiles, %d waves of %dx%d, partial sums>", KS, KS, BM,
                                                BN, NW, 32 * RB, 32 * CB);
    kgh::g_lastConvKernel = name.c_str();
    run<false, true>(x, cinStride, cinPad, cout, w + (size_t)KS * KS * cout * cinPad, g, epi, partChunks, stream);
  }
};

// The tile shapes: (variant, kernel size, row blocks and column blocks of 32
// per wave, row waves, column waves, ring depth).
#define KGH_STREAM_TILES(X)                                  \
  X(CONV_STREAM3_32, 3, 1, 1, 1, 2, 9)                       \
  X(CONV_STREAM3_64, 3, 1, 1, 2, 2, 9)                       \
  X(CONV_STREAM3_128, 3, 2, 1, 2, 2, 9)                      \
  X(CONV_STREAM3_192, 3, 3, 1, 2, 2, 3)                      \
  X(CONV_STREAM1_32, 1, 1, 1, 1, 2, 6)                       \
  X(CONV_STREAM1_64, 1, 1, 1, 2, 2, 6)

}  // namespace

namespace kgh {

bool streamFits(int variant, int cinStride, int cinPad, int cout, BoardGeom g, const ConvEpilogue<half_t>& epi) {
#define X(V, ...) \
  if(variant == V) return Stream<__VA_ARGS__>::fits(cinStride, cinPad, cout, g, epi);
  KGH_STREAM_TILES(X)
#undef X
  return false;
}

void launchStream(int variant, const half_t* x, int cinStride, int cinPad, int cout, const half_t* w, BoardGeom g,
                  const ConvEpilogue<half_t>& epi, hipStream_t stream) {
  switch(variant) {
#define X(V, ...) \
  case V: Stream<__VA_ARGS__>::launch(x, cinStride, cinPad, cout, w, g, epi, stream); return;
    KGH_STREAM_TILES(X)
#undef X
    default: throw KghError(5, "conv: not a streamed variant");
  }
}

// 3x3: the smallest tile whose workgroups fit the 256 CUs one to a CU (what
// such a launch takes is one wave's chain of K steps), else 128-row tiles
// where two workgroups' LDS fits a CU (up to 192 channels at 19x19), else 192
// rows (up to 320). us per launch with 32 / 64 / 128 / 192 rows, 192 -> 192
// channels at 19x19: one board 9.0 / 9.5 / 11.5 / 14.5; 8 boards 11.6 / 9.8 /
// 11.7 / 14.7; 16 boards 13.7 / 13.6 / 12.1 / 14.8; 32 boards 20.6 / 19.3 /
// 19.5 / 16.5; 96 boards 44.7 / 38.9 / 35.5 / 42.1; 256 -> 256 channels, 160
// boards: 97.9 / 89.2 / 87.4 / 80.4. Where two workgroups of 192 rows fit too
// (up to 144 channels), they are taken if their rounds of the CUs' 512 places
// take fewer rows (64 -> 64, sixteen convs per forward: 192 boards, 1 against 2
// rounds, 394 and 418; 160 boards, 1 and 1, 363 and 329; 128 -> 128, 96 boards,
// 1 and 2, 442 and 468; 160 boards, 2 and 2, 655 and 626).
int streamTile3x3(int cinStride, int cinPad, int cout, BoardGeom g, const ConvEpilogue<half_t>& epi) {
  const long M = (long)g.batch * g.H * g.W;
  const std::pair<int, int> tiles[] = {{CONV_STREAM3_32, 32}, {CONV_STREAM3_64, 64}, {CONV_STREAM3_128, 128}, {CONV_STREAM3_192, 192}};
  for(const auto& t : tiles)
    if((M + t.second - 1) / t.second * (cout / 64) <= 256 && streamFits(t.first, cinStride, cinPad, cout, g, epi)) return t.first;
  const bool fits192 = streamFits(CONV_STREAM3_192, cinStride, cinPad, cout, g, epi);
  if(streamFits(CONV_STREAM3_128, cinStride, cinPad, cout, g, epi) && streamLdsBytes<3, 128, 4>(cinPad, g.W) <= STREAM_MAX_LDS / 2) {
    auto roundRows = [&](int rows) { return ((M + rows - 1) / rows * (cout / 64) + 511) / 512 * rows; };
    const bool two192 = fits192 && streamLdsBytes<3, 192, 4>(cinPad, g.W) <= STREAM_MAX_LDS / 2;
    return two192 && roundRows(192) < roundRows(128) ? CONV_STREAM3_192 : CONV_STREAM3_128;
  }
  if(fits192) return CONV_STREAM3_192;
  return CONV_AUTO;
}

// The 32-row tile while its workgroups fit the 256 CUs one to a CU, else 64
// rows (streamTile3x3 has both tiles' times).
void launchStreamParts(const half_t* x, int cinStride, int cinPad, int cout, const half_t* w, BoardGeom g, const ConvEpilogue<half_t>& epi,
                       int partChunks, hipStream_t stream) {
  const long M = (long)g.batch * g.H * g.W;
  if((M + 31) / 32 * (cout / 64) > 256)
    Stream<3, 1, 1, 2, 2, 9>::launchParts(x, cinStride, cinPad, cout, w, g, epi, partChunks, stream);
  else
    Stream<3, 1, 1, 1, 2, 9>::launchParts(x, cinStride, cinPad, cout, w, g, epi, partChunks, stream);
}

// 1x1: below 24 row tiles of 192 while the 32 x 64 tiles times K, what they
// re-read of rows and weights, stay below a million (t12d384h6 at four
// boards, forwards 742 -> 652 us; against the 192-row DMA tiles, us of four convs
// per forward: 1024 -> 1024 at four boards, 0.75 M, -7; 2048 -> 768 at three,
// 0.84 M, -16; 768 -> 768 at eight, 0.84 M, +8; 768 -> 2304 at four, 1.3 M,
// +21, at eight, 2.5 M, +58; 768 -> 4096 gated at eight, 4.5 M, +237). From
// there on the DMA kernel takes gated outputs and
// K = 1024 (t12d384h6 at 16 boards); else the line follows K. Up to 192 input
// channels the streamed kernel is faster at every size: a tile holds all of K
// in little LDS, many workgroups share a CU, and the residual's load hides
// behind the others' work (192 -> 384 with a residual against the DMA tiles,
// us per forward of 17 of them: 80 boards -119, 128 -41, 160 -301, 256 -43; 512
// boards 13x13 -125; 128 -> 256, 192 boards, four of them -43). Above, its
// columns' re-reads of the rows grow with K: up to 4400 tiles (384 -> 192: 128
// boards, 4332 tiles, -40 of 18; 160 boards, 5415, +52; 256 -> 512, 48 boards,
// 4336, -4 of four; 64 boards, 5776, +8), and up to 2200 with a masked residual,
// which is read in the epilogue (384 -> 384 of t12d384h6, 12 of them against the
// 192-row DMA tiles: 24 boards, 1626 tiles, -10; 32 boards, 2166, +3; 40 boards,
// 2712, +21; 64 boards, 4332, +30). 64-row tiles for K <= 192 once the 32-row
// tiles number more than two per CU: half the weight reads.
int streamTile1x1(int cinStride, int cinPad, int cout, BoardGeom g, const ConvEpilogue<half_t>& epi) {
  const long M = (long)g.batch * g.H * g.W;
  const long tiles = (M + 31) / 32 * (cout / 64);
  if(M < 24L * 192) {
    if(tiles * cinPad > 1000000) return CONV_AUTO;
  }
  else {
    if(epi.glu || cinPad > 384 || tiles > (epi.maskResidualAdd ? 2200 : cinPad > 192 ? 4400 : LONG_MAX)) return CONV_AUTO;
  }
  const int v = cinPad <= 192 && tiles > 512 ? CONV_STREAM1_64 : CONV_STREAM1_32;
  return streamFits(v, cinStride, cinPad, cout, g, epi) ? v : CONV_AUTO;
}

void prepareFragWeights(const float* dW, half_t* dOut, int cout, int cin, int cinPad, int ks, hipStream_t stream) {
  const long total = (long)ks * ks * cout * cinPad;
  hipLaunchKernelGGL(prepareFragWeightsKernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, dW, dOut, cout, cin, cinPad, ks);
  KGH_CHECK_LAUNCH();
}

}  // namespace kgh
