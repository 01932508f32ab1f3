// Row-path kernels of some lengths (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct ZPass<70, 1>;
template struct ZPass<72, 1>;
template struct ZPass<75, 1>;
template struct RowPass<70, 1>;
template struct RowPass<72, 1>;
template struct RowPass<75, 1>;
}  // namespace jrx
