// Streaming tile GEMM on bf16 tiles: the layouts whose operands are both
// contiguous in a direction that a matmul or its gradients meet.
#include "ej_stream.h"

namespace ej {
extern template int launch_stream_m<uint16_t, kStreamKC, kStreamKC>(
    const void *, const void *, void *, const PairSrc &, const GemmGeom &, int64_t, hipStream_t);
extern template int launch_stream_m<uint16_t, kStreamFC, kStreamFC>(
    const void *, const void *, void *, const PairSrc &, const GemmGeom &, int64_t, hipStream_t);

int launch_stream_bf16(int amode, int bmode, const void *A, const void *B, void *C,
                     const PairSrc &src, GemmGeom g, int64_t n_seg, hipStream_t stream) {
  if (amode == kStreamKC && bmode == kStreamFC)
    return launch_stream_m<uint16_t, kStreamKC, kStreamFC>(A, B, C, src, g, n_seg, stream);
  if (amode == kStreamKC && bmode == kStreamKC)
    return launch_stream_m<uint16_t, kStreamKC, kStreamKC>(A, B, C, src, g, n_seg, stream);
  if (amode == kStreamFC && bmode == kStreamFC)
    return launch_stream_m<uint16_t, kStreamFC, kStreamFC>(A, B, C, src, g, n_seg, stream);
  return launch_stream_gs<uint16_t>(A, B, C, src, g, n_seg, stream);
}
}  // namespace ej
