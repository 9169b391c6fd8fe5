#include "generic_columns.h"

namespace ash {
template void gen_column_S<2>(float2*, const Tables&, const Geom&, const DftMat&, const ColDesc&, hipStream_t);
template void gen_column_S<4>(float2*, const Tables&, const Geom&, const DftMat&, const ColDesc&, hipStream_t);
}  // namespace ash
