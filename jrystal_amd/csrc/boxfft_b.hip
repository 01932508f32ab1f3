// Full-box kernels of some lengths (see boxfft_kernels.h).
#define JRX_BOXFFT_KERNELS
#include "boxfft_kernels.h"

namespace jrx {
template struct BoxPlane<54>;
template struct BoxPlane<56>;
template struct BoxPlane<60>;
template struct BoxPlane<63>;
template struct BoxPlane<64>;
template struct BoxPlane<70>;
template struct BoxPlane<72>;
template struct BoxPlane<75>;
template struct BoxPlane<80>;
template struct BoxLine<54>;
template struct BoxLine<56>;
template struct BoxLine<60>;
template struct BoxLine<63>;
template struct BoxLine<64>;
template struct BoxLine<70>;
template struct BoxLine<72>;
template struct BoxLine<75>;
template struct BoxLine<80>;
}  // namespace jrx
