// Row-path kernels of some box sides (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct RowPath<80, 1>;
template struct RowPath<128, 0>;
template struct RowPath<128, 2>;
}  // namespace jrx
