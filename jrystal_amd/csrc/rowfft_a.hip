// Row-path kernels of some box sides (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct RowPath<32, 1>;
template struct RowPath<32, 2>;
template struct RowPath<35, 1>;
template struct RowPath<36, 1>;
template struct RowPath<40, 1>;
template struct RowPath<42, 1>;
template struct RowPath<45, 1>;
}  // namespace jrx
