// Row-path kernels of some box sides (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct RowPath<70, 1>;
template struct RowPath<72, 1>;
template struct RowPath<75, 1>;
}  // namespace jrx
