// Phi with one nonzero per lane (phi_cols.hip)
#pragma once

#include "kernels_common.hpp"

namespace alto {

// ranks for which this kernel is the faster one, by pim as in
// phi_device_cached
bool phi_cols_rank(int R, int pim);

// doubles of the product cache for nnz nonzeros of rank R in this kernel's
// layout
uint64_t phi_cols_cache(uint64_t nnz, int R);

// a: the mode's stream arguments (out cleared by the caller); pim as in
// phi_device_cached
int launch_phi_cols(StreamArgs<double, double, double>& a, int pw, const double* B, double eps, double* pc, int pim,
                    hipStream_t s);

}  // namespace alto
