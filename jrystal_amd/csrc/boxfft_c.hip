// Full-box kernels of some lengths (see boxfft_kernels.h).
#define JRX_BOXFFT_KERNELS
#include "boxfft_kernels.h"

namespace jrx {
template struct BoxLine<81>;
template struct BoxLine<84>;
template struct BoxLine<90>;
template struct BoxLine<96>;
template struct BoxLine<98>;
template struct BoxLine<100>;
template struct BoxLine<105>;
template struct BoxLine<108>;
template struct BoxLine<112>;
template struct BoxLine<120>;
template struct BoxLine<126>;
template struct BoxLine<128>;
}  // namespace jrx
