// Streaming tile GEMM on bf16 tiles, the layout of one gradient of a matmul.
#include "ej_stream.h"

namespace ej {
template int launch_stream_m<uint16_t, kStreamFC, kStreamFC>(
    const void *, const void *, void *, const PairSrc &, const GemmGeom &, int64_t, hipStream_t);
}  // namespace ej
