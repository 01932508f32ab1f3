// Row-path kernels of some lengths (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct ZPass<60, 1>;
template struct ZPass<63, 1>;
template struct ZPass<64, 0>;
template struct ZPass<64, 1>;
template struct ZPass<64, 2>;
template struct ZPass<64, 3>;
template struct RowPass<60, 1>;
template struct RowPass<63, 1>;
template struct RowPass<64, 0>;
template struct RowPass<64, 1>;
template struct RowPass<64, 2>;
template struct RowPass<64, 3>;
}  // namespace jrx
