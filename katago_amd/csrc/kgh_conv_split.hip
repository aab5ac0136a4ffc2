// fp32 convolutions on the bf16 matrix cores (convSplitKernel) and their
// weight layout.
#include "kgh_conv_device.h"
#include "kgh_conv_split.h"

#include <algorithm>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------------------
// fp32 1x1 and 3x3 convolution, every batch size. An fp32 number is the sum of
// three bf16 numbers to within 2^-27 of itself (each the rounded rest of the
// ones before), so a product is the sum of nine bf16 products, of which the
// three of 2^-27 and less are left out; the six others are one
// v_mfma_f32_32x32x16_bf16 each. That is 6 x 32 cycles of the matrix core for
// 16 channels of a 32 x 32 block where v_mfma_f32_32x32x2_f32 takes 8 x 64.
// The leading product has fp32 accumulators of its own and the five small ones
// share a second set, so a sum is rounded at its own magnitude once per 16
// channels.
//
// A finite number that rounds to a bf16 infinity has the largest bf16 number as
// its first piece, and an infinity has only a third, so that it meets one piece
// of the other factor, the one with that factor's sign: sums are infinite or NaN
// as they are in fp32 (but NaN where both factors are infinite, and a finite sum
// within 2^-8 of the largest float may already be infinite). A wave that sees
// such a number splits its part of the panel a second time; looking for them
// costs 2 us of b6c96's 187 at eight boards, 10 of b18c384nbt's 1323 at one and
// 8 of its 2760 at 16 (in the first pass, without a second, 20 to 25 of each).
//
// K (16-channel chunk outer, tap inner) is cut into four groups of whole
// chunks, summed ((p0 + p1) + p2) + p3, by four waves at once or by one wave
// one group after the other; so a row rounds the same way whatever the tile,
// the LDS panel and the batch.
//
// A workgroup's input rows (its output rows and, for 3x3, one board row and
// one position either side) are loaded once, split, and kept in LDS as three
// pieces, a panel of some chunks of each group at a time; weights are split
// when they are prepared and each wave streams its fragments, 1 KB runs, from
// L2 through a ring of registers. LDS rows hold the three 32-byte pieces of
// each chunk of the panel and a 16-byte gap, an odd number of 16-byte groups: the rows of a ds_read_b128
// phase fall in distinct banks. A tap that leaves the board reads a row of
// zeros.
//
// What bounds it: up to a workgroup per CU, the chain window load (one memory
// round trip), split, products, sum, store, of which the products are a third;
// at 64 boards they are 0.45 of the time. us per launch against 32 x 32 blocks
// of v_mfma_f32_32x32x2_f32, 192 -> 192 channels at 19x19: 1 board 17.5 ->
// 15.3, 16 boards 59 -> 29, 64 boards 183 -> 92. Errors against float64, in the
// 2-norm: of one conv 0.5e-7 to 1.7e-7 (numpy's fp32 sums 1.2e-7 to 3.6e-7); of
// b18c384nbt's outputs at 16 boards, the worst one, 4.7e-7 to 6.7e-7 over five
// seeds, 2.1e-6 to 2.4e-6 on v_mfma_f32_32x32x2_f32.
constexpr int SPLIT_GROUPS = 4;
constexpr int SPLIT_STAGE_BYTES = 32 * CONV_STAGE_LD * 4;  // a wave's epilogue stage
constexpr int SPLIT_PART_BYTES = 16 * 64 * 4;              // a wave's partial sums of one 32 x 32 block
constexpr int SPLIT_MAX_LDS = 160 * 1024;

// Division by multiplication: v / d for every v with 4 v d < 2^32.
__device__ __forceinline__ unsigned splitDiv(unsigned v, unsigned magic) { return __umulhi(v << 1, magic); }
inline unsigned splitMagic(unsigned d) { return (unsigned)((0x100000000ull + 2ull * d - 1) / (2ull * d)); }

struct SplitDims {
  int panel;   // chunks of each group per LDS panel
  int panels;  // panels per group
  unsigned perMagic, groupMagic;  // 8-channel slots per window row, and per group of one
  unsigned hwMagic, wMagic;
  int colTiles;
};

constexpr float BF16_MAX = 0x1.fep127f, BF16_INF_FROM = 0x1.ffp127f;  // rounds to infinity from there

// Piece q of what the pieces before it left of a float; SPECIAL also splits
// infinities and what rounds to one.
template<bool SPECIAL>
__device__ __forceinline__ __bf16 nextPiece(int q, float rest) {
  if(SPECIAL && q < 2 && fabsf(rest) >= BF16_INF_FROM) return (__bf16)(fabsf(rest) == INFINITY ? 0.0f : copysignf(BF16_MAX, rest));
  return (__bf16)rest;
}

// The three pieces of eight floats, to dst, dst + 32 and dst + 64; or-s the
// last one's bits into seen.
template<bool SPECIAL>
__device__ __forceinline__ void storePieces(unsigned char* dst, const float4 (&v)[2], unsigned& seen) {
  float rest[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
  union {
    bf16x8 p;
    uint4 bits;
  } piece;
#pragma unroll
  for(int q = 0; q < 3; q++) {
#pragma unroll
    for(int j = 0; j < 8; j++) {
      piece.p[j] = nextPiece<SPECIAL>(q, rest[j]);
      rest[j] -= (float)piece.p[j];
    }
    *(uint4*)(dst + q * 32) = piece.bits;
  }
  seen |= piece.bits.x | piece.bits.y | piece.bits.z | piece.bits.w;
}
// What is or rounds to an infinity leaves a NaN in the last piece, whose
// exponent has its highest bit set; so have third pieces of 2 and more, of
// numbers from 2^18, which are split the same way again.
__device__ __forceinline__ bool anySpecial(unsigned seen) { return __any(seen & 0x40004000u); }

// One K step of RB row blocks: six products each. A piece's registers take
// the next step's right after its last use here (a step starts with the piece
// that is free first), and a weight piece's those of the step a ring ahead.
// Left to itself the compiler moves every load down to its use.
template<int RB, typename NextA, typename NextB>
__device__ __forceinline__ void splitStep(floatx16 (&lead)[RB], floatx16 (&small)[RB], bf16x8 (&a)[RB][3], bf16x8 (&b)[3], NextA&& nextA,
                                          NextB&& nextB) {
  constexpr int PA[6] = {0, 0, 0, 1, 1, 2}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
  for(int i = 0; i < 6 * RB; i++) {
    const int p = i / RB, rb = i % RB;
    if(p == 0) lead[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[rb][0], b[0], lead[rb], 0, 0, 0);
    else small[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[rb][PA[p]], b[PB[p]], small[rb], 0, 0, 0);
    if(p == 2 || p == 4 || p == 5) nextA(a[rb][PA[p]], rb, PA[p]);
    if(rb == RB - 1 && p == 2) nextB(b[2], 2);
    if(rb == RB - 1 && p == 4) nextB(b[1], 1);
    if(rb == RB - 1 && p == 5) nextB(b[0], 0);
    __builtin_amdgcn_sched_barrier(0);
  }
}

template<int RB>
__device__ __forceinline__ void clearTiles(floatx16 (&t)[RB]) {
#pragma unroll
  for(int rb = 0; rb < RB; rb++)
#pragma unroll
    for(int r = 0; r < 16; r++) t[rb][r] = 0.0f;
}

// Wave (wn, wk) of WN x 4 computes 32 RB rows x 32 columns of group wk.
template<int KS, int RB, int WN, bool GLU>
__global__ __launch_bounds__(64 * WN * SPLIT_GROUPS, 1) void convSplitKernel(const float* __restrict__ x, int cinStride, int cinPad, int cout,
                                                                   const __bf16* __restrict__ wf, BoardGeom g, SplitDims sd,
                                                                   ConvEpilogue<float> epi) {
  constexpr int KW = SPLIT_GROUPS;
  constexpr int NT = 64 * WN * KW;
  constexpr int BM = 32 * RB;
  constexpr int TAPS = KS * KS;
  constexpr int DEPTH = KS == 3 ? 3 : 4;
  extern __shared__ __attribute__((aligned(1024))) unsigned char splitLds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN;
  const int wk = wave / WN;
  const int laneRow = lane & 31;
  const int kq = lane >> 5;
  const int HW = g.H * g.W;
  const int M = g.batch * HW;
  const int tile = xcdContiguousTile();
  const int rowTile = tile / sd.colTiles;
  const int m0 = rowTile * BM;
  const int n0 = (tile - rowTile * sd.colTiles) * 32 * WN;
  const int halo = KS == 3 ? g.W + 1 : 0;
  const int winRows = BM + 2 * halo;
  const int rowB = KW * sd.panel * 96 + 16;
  float* rowScale = (float*)splitLds;
  unsigned char* win = splitLds + (KS == 1 ? BM * 4 : 0);

  const int chunks = cinPad / 16;
  const int nBlocks = cout / 32;
  const unsigned laneOff = lane * 16;
  auto readB = [&](int s, int piece) {
    return *(const bf16x8*)((const char*)wf + ((size_t)s * nBlocks + n0 / 32 + wn) * 3072 + laneOff + piece * 1024);
  };
  auto groupStart = [&](unsigned gr) { return (int)(gr * (unsigned)chunks / SPLIT_GROUPS); };

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

  // LDS byte address of the lane's A fragments per tap (channel 0 of the
  // wave's part of the panel and its k group, first piece).
  int aAddr[RB][TAPS];
  const int sp0 = m0 % HW;
#pragma unroll
  for(int rb = 0; rb < RB; rb++) {
    const int r = rb * 32 + laneRow;
    const int inRow = wk * sd.panel * 96 + kq * 16;
    if constexpr(KS == 3) {
      const unsigned v = sp0 + r;
      const int sp = v - splitDiv(v, sd.hwMagic) * HW;
      const int y = splitDiv(sp, sd.wMagic);
      const int xx = sp - y * g.W;
      const bool live = m0 + r < M;
      const bool yOk[3] = {live && y > 0, live, live && y < g.H - 1};
      const bool xOk[3] = {xx > 0, true, xx < g.W - 1};
      const int base = (r + halo) * rowB + inRow;
#pragma unroll
      for(int t = 0; t < 9; t++)
        aAddr[rb][t] = yOk[t / 3] && xOk[t % 3] ? base + ((t / 3 - 1) * g.W + t % 3 - 1) * rowB : winRows * rowB + inRow;
    }
    else {
      aAddr[rb][0] = r * rowB + inRow;
    }
  }
  if constexpr(KS == 3) {
    for(int i = tid * 16; i < rowB; i += NT * 16) *(uint4*)(win + winRows * rowB + i) = make_uint4(0, 0, 0, 0);
  }

  // Splits chunks first .. first + panel - 1 of every group into LDS. A thread has eight 16-byte loads in flight. Rows outside [0, M) only
  // feed taps that read zeros, or outputs that are never stored: they load a
  // valid address, as do the slots past the last row or the group's last
  // chunk, which are not written.
  auto loadPanel = [&](int first, auto specialTag) {
    constexpr bool SPECIAL = decltype(specialTag)::value;
    constexpr int U = SPECIAL ? 1 : 4;
    unsigned seen = 0;
    const int groupSlots = sd.panel * 2;
    const int per = KW * groupSlots;
    const int total = winRows * per;
    for(int base = 0; base < total; base += U * NT) {
      float4 val[U][2];
      int dst[U];
#pragma unroll
      for(int u = 0; u < U; u++) {
        const unsigned slot = base + u * NT + tid;
        const unsigned row = splitDiv(slot, sd.perMagic);
        const unsigned at = slot - __umul24(row, per);
        const unsigned k = splitDiv(at, sd.groupMagic);
        const int ch = (groupStart(k) + first) * 16 + (int)(at - __umul24(k, groupSlots)) * 8;
        const bool live = (int)slot < total && ch < groupStart(k + 1) * 16;
        const int gm = min(max(m0 - halo + (int)row, 0), M - 1);
        const float4* src = (const float4*)(x + (size_t)gm * cinStride + (live ? ch : 0));
        val[u][0] = src[0];
        val[u][1] = src[1];
        dst[u] = live ? (int)(__umul24(row, rowB) + __umul24(at >> 1, 96) + (at & 1) * 16) : -1;
      }
#pragma unroll
      for(int u = 0; u < U; u++)
        if(dst[u] >= 0) storePieces<SPECIAL>(win + dst[u], val[u], seen);
    }
    return seen;
  };

  floatx16 lead[RB], small[RB], sum[RB];
  clearTiles(lead);
  clearTiles(small);
  auto readA = [&](int tap, int c, int rb, int piece) { return *(const bf16x8*)(win + aAddr[rb][tap] + c * 96 + piece * 32); };
  bf16x8 a[RB][3], bRing[DEPTH][3];
  for(int first = 0; first < sd.panel * sd.panels; first += sd.panel) {
    // This wave's steps of the panel.
    const int c0 = groupStart(wk) + first;
    const int pc = min(max(groupStart(wk + 1) - c0, 0), sd.panel);
    const int s0 = min(c0, chunks - 1) * TAPS;
    const int sLast = max(pc * TAPS - 1, 0);
#pragma unroll
    for(int d = 0; d < DEPTH; d++)
#pragma unroll
      for(int q = 0; q < 3; q++) bRing[d][q] = readB(s0 + min(d, sLast), q);
    if(first > 0) __syncthreads();  // every wave is done with the panel before
    if(__builtin_expect(anySpecial(loadPanel(first, std::false_type())), 0)) loadPanel(first, std::true_type());
    __syncthreads();
    if(pc == 0) continue;
#pragma unroll
    for(int rb = 0; rb < RB; rb++)
#pragma unroll
      for(int q = 0; q < 3; q++) a[rb][q] = readA(0, 0, rb, q);
    // Reads past the last step repeat one of the panel.
    if constexpr(KS == 3) {
      for(int c = 0; c < pc; c++) {
#pragma unroll
        for(int t = 0; t < 9; t++)
          splitStep(
            lead, small, a, bRing[t % DEPTH],
            [&](bf16x8& f, int rb, int q) { f = t < 8 ? readA(t + 1, c, rb, q) : readA(0, min(c + 1, pc - 1), rb, q); },
            [&](bf16x8& f, int q) { f = readB(s0 + min(9 * c + t + DEPTH, sLast), q); });
      }
    }
    else {
      for(int i = 0; i < pc; i += DEPTH) {
#pragma unroll
        for(int d = 0; d < DEPTH; d++)
          if(i + d < pc)
            splitStep(
              lead, small, a, bRing[d], [&](bf16x8& f, int rb, int q) { f = readA(0, min(i + d + 1, pc - 1), rb, q); },
              [&](bf16x8& f, int q) { f = readB(s0 + min(i + d + DEPTH, sLast), q); });
      }
    }
  }
#pragma unroll
  for(int rb = 0; rb < RB; rb++) sum[rb] = lead[rb] + small[rb];

  // The waves' sums meet in LDS; wave w finishes block w of the RB x WN.
  __syncthreads();
  float* part = (float*)win;
#pragma unroll
  for(int rb = 0; rb < RB; rb++)
#pragma unroll
    for(int r = 0; r < 16; r++) part[(((wk * RB + rb) * WN + wn) * 16 + r) * 64 + lane] = sum[rb][r];
  __syncthreads();
  static_assert(RB * WN <= WN * KW, "a wave per block");
  if(wave >= RB * WN) return;
  floatx16 total[1][1];
#pragma unroll
  for(int r = 0; r < 16; r++) {
    float v[KW];
#pragma unroll
    for(int k = 0; k < KW; k++) v[k] = part[((k * RB * WN + wave) * 16 + r) * 64 + lane];
    total[0][0][r] = ((v[0] + v[1]) + v[2]) + v[3];
  }
  float* stage = part + (KW * RB * WN * SPLIT_PART_BYTES + wave * SPLIT_STAGE_BYTES) / 4;
  const int rb = wave / WN;
  storeWaveEpilogue<float, 1, 1, false, GLU, KS == 1, KS == 1>(total, stage, m0 + rb * 32, n0 + wn * 32, M, HW, epi,
                                                              rowNorm ? rowScale + rb * 32 : nullptr);
}

// 1x1, many rows: the waves of a workgroup take a 32-column block each and all
// of K, so that the rows, loaded and split once, serve up to 256 columns (with
// 64 columns, splitting takes 0.4 of the time of the products). A wave folds
// its accumulators at the end of each K group, in the order of the kernel
// above.
struct SplitWideDims {
  int panel;          // chunks per LDS panel
  unsigned perMagic;  // 8-channel slots per row
  int parts;          // workgroups per row tile
};

template<bool GLU>
__global__ __launch_bounds__(512, 2) void convSplitWideKernel(const float* __restrict__ x, int cinStride, int cinPad, int cout,
                                                              const __bf16* __restrict__ wf, int M, int HW, SplitWideDims sd,
                                                              ConvEpilogue<float> epi) {
  constexpr int BM = 32;
  constexpr int DEPTH = 4;
  extern __shared__ __attribute__((aligned(1024))) unsigned char splitLds[];
  const int NT = blockDim.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = xcdContiguousTile();
  const int rowTile = tile / sd.parts;
  const int m0 = rowTile * BM;
  const int nBlocks = cout / 32;
  const int block = (tile - rowTile * sd.parts) * (NT / 64) + wave;
  const bool live = block < nBlocks;  // the last part may have fewer blocks than waves
  const int rowB = sd.panel * 96 + 16;
  float* rowScale = (float*)splitLds;
  unsigned char* win = splitLds + BM * 4;
  const int chunks = cinPad / 16;
  const unsigned laneOff = lane * 16;
  auto readB = [&](int s, int piece) {
    return *(const bf16x8*)((const char*)wf + ((size_t)s * nBlocks + min(block, nBlocks - 1)) * 3072 + laneOff + piece * 1024);
  };
  const bool rowNorm = epi.rowNormIn != nullptr;
  if(rowNorm) {
    for(int i = tid; i < BM; i += NT) {
      float nq[KGH_NORM_MAX_BLOCKS], nMask = 0.0f;
      const bool in = m0 + i < M;
      if(in) kgh_row_norm_load(epi, m0 + i, nq, nMask);
      rowScale[i] = in ? kgh_row_norm_finish(epi, nq, nMask) : 0.0f;
    }
  }
  const unsigned char* aRow = win + (lane & 31) * rowB + (lane >> 5) * 16;
  auto readA = [&](int c, int piece) { return *(const bf16x8*)(aRow + c * 96 + piece * 32); };

  floatx16 lead[1], small[1], sum[1];
  clearTiles(lead);
  clearTiles(small);
  clearTiles(sum);
  int group = 0;
  bf16x8 a[1][3], bRing[DEPTH][3];
  for(int c0 = 0; c0 < chunks; c0 += sd.panel) {
    const int pc = min(sd.panel, chunks - c0);
#pragma unroll
    for(int d = 0; d < DEPTH; d++)
#pragma unroll
      for(int q = 0; q < 3; q++) bRing[d][q] = readB(c0 + min(d, pc - 1), q);
    if(c0 > 0) __syncthreads();  // every wave is done with the panel before
    auto loadPanel = [&](auto specialTag) {
      constexpr bool SPECIAL = decltype(specialTag)::value;
      constexpr int U = SPECIAL ? 1 : 4;
      unsigned seen = 0;
      const int per = sd.panel * 2;
      const int total = BM * per;
      for(int base = 0; base < total; base += U * NT) {
        float4 val[U][2];
        int dst[U];
#pragma unroll
        for(int u = 0; u < U; u++) {
          const unsigned slot = base + u * NT + tid;
          const unsigned row = splitDiv(slot, sd.perMagic);
          const unsigned at = slot - __umul24(row, per);
          const bool in = (int)slot < total && (int)at < pc * 2;
          const int gm = min(m0 + (int)row, M - 1);
          const float4* src = (const float4*)(x + (size_t)gm * cinStride + (in ? c0 * 16 + at * 8 : 0));
          val[u][0] = src[0];
          val[u][1] = src[1];
          dst[u] = in ? (int)(__umul24(row, rowB) + __umul24(at >> 1, 96) + (at & 1) * 16) : -1;
        }
#pragma unroll
        for(int u = 0; u < U; u++)
          if(dst[u] >= 0) storePieces<SPECIAL>(win + dst[u], val[u], seen);
      }
      return seen;
    };
    if(__builtin_expect(anySpecial(loadPanel(std::false_type())), 0)) loadPanel(std::true_type());
    __syncthreads();
    if(!live) continue;
#pragma unroll
    for(int q = 0; q < 3; q++) a[0][q] = readA(0, q);
    for(int i = 0; i < pc; i += DEPTH) {
#pragma unroll
      for(int d = 0; d < DEPTH; d++) {
        if(i + d < pc) {
          splitStep(
            lead, small, a, bRing[d], [&](bf16x8& f, int, int q) { f = readA(min(i + d + 1, pc - 1), q); },
            [&](bf16x8& f, int q) { f = readB(c0 + min(i + d + DEPTH, pc - 1), q); });
          while(group < SPLIT_GROUPS && (group + 1) * chunks / SPLIT_GROUPS <= c0 + i + d + 1) {  // groups of no chunk too
            sum[0] += lead[0] + small[0];
            clearTiles(lead);
            clearTiles(small);
            group++;
          }
        }
      }
    }
  }
  __syncthreads();  // every wave is done with the window before it holds the stages
  if(!live) return;
  floatx16 out[1][1] = {{sum[0]}};
  storeWaveEpilogue<float, 1, 1, false, GLU, true, true>(out, (float*)(win + wave * SPLIT_STAGE_BYTES), m0, block * 32, M, HW, epi,
                                                         rowNorm ? rowScale : nullptr);
}

// The split weights: for each (16-channel chunk, tap, 32-column block, piece)
// 64 lanes x 8 channels, lane l = column l % 32, channels 8 (l / 32) .. + 7: a
// wave's fragment is one contiguous 1 KB run.
__global__ void prepareSplitWeightsKernel(const float* __restrict__ src, __bf16* __restrict__ dst, int cout, int cin, int cinPad, int ks) {
  const int taps = ks * ks;
  const long total = (long)taps * cout * cinPad;
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if(idx >= total) return;
  const int lane = (int)(idx >> 3) & 63;
  const long blk = idx >> 9;
  const int nb = (int)(blk % (cout / 32));
  const long step = blk / (cout / 32);
  const int tap = (int)(step % taps);
  const int oc = nb * 32 + (lane & 31);
  const int ic = (int)(step / taps) * 16 + (lane >> 5) * 8 + (int)(idx & 7);
  float rest = ic < cin ? src[(((size_t)oc * cin + ic) * ks + tap / ks) * ks + tap % ks] : 0.0f;
  for(int q = 0; q < 3; q++) {
    const __bf16 p = nextPiece<true>(q, rest);
    dst[blk * 1536 + q * 512 + (idx & 511)] = p;
    rest -= (float)p;
  }
}

// Rows of a window (and the row of zeros), and the bytes of one.
long splitWindowRows(int ks, int rows, int W) { return rows + (ks == 3 ? 2 * (W + 1) + 1 : 0); }
int splitRowBytes(int panel) { return SPLIT_GROUPS * panel * 96 + 16; }

template<int KS, int RB, int WN>
void launchTile(const float* x, int cinStride, int cinPad, int cout, const __bf16* wf, BoardGeom g, const ConvEpilogue<float>& epi,
                hipStream_t stream) {
  constexpr int BM = 32 * RB, KW = SPLIT_GROUPS;
  static const std::string name = kernelLabel("convSplitKernel<%dx%d fp32, %dx%d tiles, K over %d waves>", KS, KS, BM, 32 * WN, KW);
  kgh::g_lastConvKernel = name.c_str();
  const int M = g.batch * g.H * g.W;
  const int colTiles = cout / (32 * WN);
  const long tiles = (long)((M + BM - 1) / BM) * colTiles;
  const int rows = (int)splitWindowRows(KS, BM, g.W);
  const int fixed = KS == 1 ? BM * 4 : 0;
  const int sums = KW * RB * WN * SPLIT_PART_BYTES + RB * WN * SPLIT_STAGE_BYTES;
  // The largest panel in the LDS of a CU, or in half of it where there are two
  // workgroups to a CU and the sums leave room for both: one loads and splits
  // while the other multiplies.
  const int budget = (tiles <= 256 || RB > 1 ? SPLIT_MAX_LDS : SPLIT_MAX_LDS / 2) - fixed;
  const int group = (cinPad / 16 + SPLIT_GROUPS - 1) / SPLIT_GROUPS;  // chunks of the longest
  const int most = std::max((budget / rows - 16) / (96 * KW), 1);
  const int panels = (group + most - 1) / most;
  const int panel = (group + panels - 1) / panels;
  const int lds = fixed + std::max(rows * splitRowBytes(panel), sums);
  if(lds > SPLIT_MAX_LDS) throw KghError(5, "conv: board too wide for the fp32 kernel");
  const SplitDims sd = {panel, panels, splitMagic(KW * panel * 2), splitMagic(panel * 2), splitMagic(g.H * g.W), splitMagic(g.W), colTiles};
  const dim3 grid((unsigned)tiles), block(64 * WN * KW);
  if constexpr(KS == 1) {
    if(epi.glu) {
      hipLaunchKernelGGL((convSplitKernel<KS, RB, WN, true>), grid, block, lds, stream, x, cinStride, cinPad, cout, wf, g, sd, epi);
      KGH_CHECK_LAUNCH();
      return;
    }
  }
  hipLaunchKernelGGL((convSplitKernel<KS, RB, WN, false>), grid, block, lds, stream, x, cinStride, cinPad, cout, wf, g, sd, epi);
  KGH_CHECK_LAUNCH();
}

void launchWide(const float* x, int cinStride, int cinPad, int cout, const __bf16* wf, BoardGeom g, const ConvEpilogue<float>& epi,
                hipStream_t stream) {
  constexpr int BM = 32;
  kgh::g_lastConvKernel = "convSplitWideKernel<1x1 fp32, 32-row tiles, up to 8 waves of 32 columns>";
  const int M = g.batch * g.H * g.W;
  const int blocks = cout / 32, parts = (blocks + 7) / 8, waves = (blocks + parts - 1) / parts;
  const int chunks = cinPad / 16;
  const int most = ((SPLIT_MAX_LDS - BM * 4) / BM - 16) / 96;
  const int panels = (chunks + most - 1) / most, panel = (chunks + panels - 1) / panels;
  const int lds = BM * 4 + std::max(BM * (96 * panel + 16), waves * SPLIT_STAGE_BYTES);
  const SplitWideDims sd = {panel, splitMagic(panel * 2), parts};
  const dim3 grid((unsigned)((long)((M + BM - 1) / BM) * parts)), block(64 * waves);
  if(epi.glu)
    hipLaunchKernelGGL((convSplitWideKernel<true>), grid, block, lds, stream, x, cinStride, cinPad, cout, wf, M, g.H * g.W, sd, epi);
  else
    hipLaunchKernelGGL((convSplitWideKernel<false>), grid, block, lds, stream, x, cinStride, cinPad, cout, wf, M, g.H * g.W, sd, epi);
  KGH_CHECK_LAUNCH();
}

}  // namespace

namespace kgh {

bool splitFits(int ks, int cinStride, int cinPad, int cout, const ConvEpilogue<float>& epi) {
  return (ks == 1 || ks == 3) && cinPad % 16 == 0 && cinStride % 4 == 0 && cout % 32 == 0 &&
         (ks == 1 || (!epi.glu && epi.rowNormIn == nullptr && epi.ropeEnd == 0));
}

// 3x3: a tile's window with one chunk of each K group in the LDS (boards up to
// 187 wide on 32-row tiles, 155 on 96), and positions of a board within the
// exact range of the divisions by multiplication.
static bool windowFits(int rows, BoardGeom g) {
  const long hw = (long)g.H * g.W;
  return splitWindowRows(3, rows, g.W) * splitRowBytes(1) <= SPLIT_MAX_LDS && 4 * (hw + 96) * hw < (1L << 32);
}
bool splitBoardFits(int ks, BoardGeom g) { return ks == 1 || windowFits(32, g); }

bool splitVariantFits(int variant, int ks, int cout, BoardGeom g) {
  if(ks == 3) {
    if(variant == CONV_SPLIT3_32) return windowFits(32, g);
    return cout % 64 == 0 && ((variant == CONV_SPLIT3_64 && windowFits(64, g)) || (variant == CONV_SPLIT3_96 && windowFits(96, g)));
  }
  return variant == CONV_SPLIT1_K || variant == CONV_SPLIT1_WIDE;
}

// 3x3: the smallest tile whose workgroups fit the 256 CUs one to a CU, else 96
// rows. us per launch with 32 / 64 / 96 rows, 192 -> 192 channels at 19x19: 1
// board 15.3 / 21.4 / 26.7, 16 boards 40.2 / 42.6 / 29.1, 64 boards 110 / 111
// / 92. Outputs that are no multiple of 64 columns keep 32 rows (96 -> 96
// channels at 8 boards: 12.0, 12.9 on 64 rows; at 64: 40, 47).
//
// 1x1: K over the waves up to two workgroups per CU, then columns over the
// waves. us per launch, K / columns: 384 <-> 192 channels 9.8 / 14.1 at one
// board, 24.8 / 21.8 at 16; t12d384h6's GEMMs 13.6 / 19.6 at one board, 44.1 /
// 32.3 at eight.
int splitChoice(int ks, int cout, BoardGeom g) {
  const long M = (long)g.batch * g.H * g.W;
  const int cols = cout % 64 == 0 ? 64 : 32;
  auto tiles = [&](int rows) { return (M + rows - 1) / rows * (cout / cols); };
  if(ks == 1) return tiles(32) > 512 ? CONV_SPLIT1_WIDE : CONV_SPLIT1_K;
  if(cols == 32 || tiles(32) <= 256 || !windowFits(96, g)) return CONV_SPLIT3_32;
  return tiles(64) <= 256 ? CONV_SPLIT3_64 : CONV_SPLIT3_96;
}

void launchSplit(int variant, const float* x, int cinStride, int cinPad, int cout, const float* w, BoardGeom g,
                 const ConvEpilogue<float>& epi, hipStream_t stream) {
  const __bf16* wf = (const __bf16*)w;
  const bool cols64 = cout % 64 == 0;
  switch(variant) {
    case CONV_SPLIT3_32:
      if(cols64) launchTile<3, 1, 2>(x, cinStride, cinPad, cout, wf, g, epi, stream);
      else launchTile<3, 1, 1>(x, cinStride, cinPad, cout, wf, g, epi, stream);
      return;
    case CONV_SPLIT3_64: launchTile<3, 2, 2>(x, cinStride, cinPad, cout, wf, g, epi, stream); return;
    case CONV_SPLIT3_96: launchTile<3, 3, 2>(x, cinStride, cinPad, cout, wf, g, epi, stream); return;
    case CONV_SPLIT1_K:
      if(cols64) launchTile<1, 1, 2>(x, cinStride, cinPad, cout, wf, g, epi, stream);
      else launchTile<1, 1, 1>(x, cinStride, cinPad, cout, wf, g, epi, stream);
      return;
    case CONV_SPLIT1_WIDE: launchWide(x, cinStride, cinPad, cout, wf, g, epi, stream); return;
    default: throw KghError(5, "conv: not an fp32 tile");
  }
}

void prepareSplitWeights(const float* dW, float* dOut, int cout, int cin, int cinPad, int ks, hipStream_t stream) {
  const long total = (long)ks * ks * cout * cinPad;
  hipLaunchKernelGGL(prepareSplitWeightsKernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, dW, (__bf16*)dOut, cout, cin,
                     cinPad, ks);
  KGH_CHECK_LAUNCH();
}

}  // namespace kgh
