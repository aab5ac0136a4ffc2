// Launchers of the streamed-weight convolutions (kgh_conv_stream.hip).
#ifndef KGH_CONV_STREAM_H
#define KGH_CONV_STREAM_H

#include "kgh_common.h"

namespace kgh {

// The kernel of the calling thread's last conv launch (see lastConvKernel).
extern thread_local const char* g_lastConvKernel;

// The streamed tile (ConvVariant) the built-in choice runs for a 3x3 or 1x1
// conv of this shape, or CONV_AUTO where other kernels take it.
int streamTile3x3(int cinStride, int cinPad, int cout, BoardGeom g, const ConvEpilogue<half_t>& epi);
int streamTile1x1(int cinStride, int cinPad, int cout, BoardGeom g, const ConvEpilogue<half_t>& epi);
// Whether a streamed variant (CONV_STREAM*) takes the shape.
bool streamFits(int variant, int cinStride, int cinPad, int cout, BoardGeom g, const ConvEpilogue<half_t>& epi);
// Runs it; w are the prepared weights, the fragment layout following the first.
void launchStream(int variant, const half_t* x, int cinStride, int cinPad, int cout, const half_t* w, BoardGeom g,
                  const ConvEpilogue<half_t>& epi, hipStream_t stream);

// 3x3 with partial sums of partChunks 32-channel chunks each, added in order
// (the low-latency mode), for shapes that CONV_STREAM3_64 takes.
void launchStreamParts(const half_t* x, int cinStride, int cinPad, int cout, const half_t* w, BoardGeom g, const ConvEpilogue<half_t>& epi,
                       int partChunks, hipStream_t stream);

// fp32 weights (oc, ic, y, x) to the streamed kernels' fragment layout.
void prepareFragWeights(const float* dW, half_t* dOut, int cout, int cin, int cinPad, int ks, hipStream_t stream);

}  // namespace kgh

#endif
