// Row-path kernels of some lengths (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct ZPass<48, 1>;
template struct ZPass<49, 1>;
template struct ZPass<50, 1>;
template struct ZPass<54, 1>;
template struct ZPass<56, 1>;
template struct RowPass<48, 1>;
template struct RowPass<49, 1>;
template struct RowPass<50, 1>;
template struct RowPass<54, 1>;
template struct RowPass<56, 1>;
}  // namespace jrx
