#include "generic_columns.h"

namespace ash {
template void gen_column_S<8>(float2*, const Tables&, const Geom&, const DftMat&, const ColDesc&, hipStream_t);
}  // namespace ash
