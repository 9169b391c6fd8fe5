// Host launchers of the general-size kernels (generic.hip, its own translation unit).
#pragma once
#include "column.h"

namespace ash {

// Shape of the DFT matrix of a line axis or the column axis of length n (A and tw are
// null), and the device memory it takes.
DftMat dft_matrix_shape(int n, bool columns);
size_t dft_matrix_bytes(const DftMat& d);
// Fills A (dft_matrix_bytes on the device) from d.tw, the axis' full-length twiddle table.
void dft_matrix_fill(const DftMat& d, float4* A, hipStream_t s);

void gen_xfwd(float2* spec, const Geom& g, const DftMat& d, hipStream_t s);
void gen_xinv(int epi, float2* spec, const Tables& T, const Geom& g, const DftMat& d, const EpiDesc& e, hipStream_t s);
void gen_ypass(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const OpDesc& op, hipStream_t s);
void gen_ypower(const float2* spec, const Tables& T, const Geom& g, const DftMat& d, double2* part, hipStream_t s);
void gen_ysa(float2* spec, const Tables& T, const Geom& g, const ScreenDesc& sd, hipStream_t s);
// Column pass cd.mode on nT outside the FFT set; its blocks (one partial each for COL_MAXABS).
void gen_column(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const ColDesc& cd, hipStream_t s);
int gen_column_blocks(int ncols);
template <int S>
void gen_column_S(float2* spec, const Tables& T, const Geom& g, const DftMat& d, const ColDesc& cd, hipStream_t s);

}  // namespace ash
