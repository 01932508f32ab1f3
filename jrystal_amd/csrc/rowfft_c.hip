// Row-path kernels of some box sides (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct RowPath<60, 1>;
template struct RowPath<63, 1>;
template struct RowPath<64, 0>;
template struct RowPath<64, 1>;
template struct RowPath<64, 2>;
}  // namespace jrx
