// Launcher of the matrix-core dense kernel for fused gates of 5 and 6 targets,
// in complex128 also 3 and 4 (dense_mfma.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "device.h"

namespace qvd {

// One pass of a dense op with d.k = 5 or 6 (complex128: 3 to 6) targets over the controlled
// subspace (same descriptor as launch_dense); mat is the 2^k x 2^k matrix,
// row-major, in device memory. cus = compute units (grid size).
template <typename T2>
hipError_t launch_dense_mfma(T2 *s, const GateDesc &d, const T2 *mat, unsigned cus, hipStream_t st);

}  // namespace qvd
