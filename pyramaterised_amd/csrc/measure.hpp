// Launchers of the state-measure kernels (measure.hip) for the C ABI entry
// points in engine.hip.  Arguments are checked by the callers; workspace
// sizes come from the *_ws functions.  Not part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace pqs {

// Reduced one-qubit density matrices and Meyer-Wallach Q (pqs_mw).
size_t mw_ws(int n, int64_t batch);
int mw_launch(int dtype, const void *states, int n, int64_t batch, double *rho, double *q, void *ws, hipStream_t st);

// Stabiliser Renyi sums (pqs_magic), n <= 13.
size_t magic_ws(int n, int64_t batch);
int magic_launch(int dtype, const void *states, int n, int64_t batch, double alpha, double *out, void *ws,
                 hipStream_t st);

}  // namespace pqs
