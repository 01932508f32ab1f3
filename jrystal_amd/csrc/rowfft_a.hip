// Row-path kernels of some lengths (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct ZPass<32, 1>;
template struct ZPass<32, 2>;
template struct ZPass<35, 1>;
template struct ZPass<36, 1>;
template struct ZPass<40, 1>;
template struct ZPass<42, 1>;
template struct ZPass<45, 1>;
template struct RowPass<32, 1>;
template struct RowPass<32, 2>;
template struct RowPass<35, 1>;
template struct RowPass<36, 1>;
template struct RowPass<40, 1>;
template struct RowPass<42, 1>;
template struct RowPass<45, 1>;
}  // namespace jrx
