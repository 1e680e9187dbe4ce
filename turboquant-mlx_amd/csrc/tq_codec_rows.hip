// The streaming codec for any number of rows (d = 64, 128 and 256).
#include "tq_codec_stream.h"

namespace tqc {
template void launch_encode_rows<64, true>(const EncodeCall&);
template void launch_encode_rows<256, true>(const EncodeCall&);
template void launch_encode_rows<128, true>(const EncodeCall&);
template void launch_dequant_rows<64, true>(const DequantCall&);
template void launch_dequant_rows<256, true>(const DequantCall&);
template void launch_dequant_rows<128, true>(const DequantCall&);
}  // namespace tqc
