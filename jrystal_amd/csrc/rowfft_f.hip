// Row-path kernels of some lengths (see rowfft_kernels.h).
#define JRX_ROWFFT_KERNELS
#include "rowfft_kernels.h"

namespace jrx {
template struct RowPass<81, 1>;
template struct RowPass<84, 1>;
template struct RowPass<90, 1>;
template struct RowPass<96, 1>;
template struct RowPass<98, 1>;
template struct RowPass<100, 1>;
template struct RowPass<105, 1>;
template struct RowPass<108, 1>;
template struct RowPass<112, 1>;
template struct RowPass<120, 1>;
template struct RowPass<126, 1>;
}  // namespace jrx
