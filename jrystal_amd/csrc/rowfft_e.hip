// Row-path kernels of some lengths (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct ZPass<80, 1>;
template struct ZPass<128, 0>;
template struct ZPass<128, 2>;
template struct RowPass<80, 1>;
template struct RowPass<128, 0>;
template struct RowPass<128, 2>;
}  // namespace jrx
