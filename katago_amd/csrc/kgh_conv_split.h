// Launchers of the fp32 convolutions on bf16 matrix cores (kgh_conv_split.hip).
#ifndef KGH_CONV_SPLIT_H
#define KGH_CONV_SPLIT_H

#include "kgh_common.h"

namespace kgh {

extern thread_local const char* g_lastConvKernel;

// Whether they take a ks x ks conv, whatever its batch, and one on boards of
// this size.
bool splitFits(int ks, int cinStride, int cinPad, int cout, const ConvEpilogue<float>& epi);
bool splitBoardFits(int ks, BoardGeom g);
// Whether a tile (ConvVariant CONV_SPLIT*) takes such a conv, and the one the
// built-in choice runs. All of them give the same bits.
bool splitVariantFits(int variant, int ks, int cout, BoardGeom g);
int splitChoice(int ks, int cout, BoardGeom g);
// Runs one; w are the split weights.
void launchSplit(int variant, const float* x, int cinStride, int cinPad, int cout, const float* w, BoardGeom g,
                 const ConvEpilogue<float>& epi, hipStream_t stream);
// fp32 weights (oc, ic, y, x) to the split layout: 3/2 floats per weight.
void prepareSplitWeights(const float* dW, float* dOut, int cout, int cin, int cinPad, int ks, hipStream_t stream);

}  // namespace kgh

#endif
