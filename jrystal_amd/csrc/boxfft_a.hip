// Full-box kernels of some lengths (see boxfft_kernels.h).
#define JRX_BOXFFT_KERNELS
#include "boxfft_kernels.h"

namespace jrx {
template struct BoxPlane<32>;
template struct BoxPlane<35>;
template struct BoxPlane<36>;
template struct BoxPlane<40>;
template struct BoxPlane<42>;
template struct BoxPlane<45>;
template struct BoxPlane<48>;
template struct BoxPlane<49>;
template struct BoxPlane<50>;
template struct BoxLine<32>;
template struct BoxLine<35>;
template struct BoxLine<36>;
template struct BoxLine<40>;
template struct BoxLine<42>;
template struct BoxLine<45>;
template struct BoxLine<48>;
template struct BoxLine<49>;
template struct BoxLine<50>;
}  // namespace jrx
