// The streaming codec with levels as bytes (d = 64, 128 and 256).
#include "tq_codec_stream.h"

namespace tqc {
template void launch_encode_indices<64>(const EncodeCall&);
template void launch_encode_indices<128>(const EncodeCall&);
template void launch_encode_indices<256>(const EncodeCall&);
template void launch_dequant_indices<64>(const DequantCall&, uint32_t);
template void launch_dequant_indices<128>(const DequantCall&, uint32_t);
template void launch_dequant_indices<256>(const DequantCall&, uint32_t);
}  // namespace tqc
