// Row-path kernels of some box sides (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct RowPath<48, 1>;
template struct RowPath<49, 1>;
template struct RowPath<50, 1>;
template struct RowPath<54, 1>;
template struct RowPath<56, 1>;
}  // namespace jrx
