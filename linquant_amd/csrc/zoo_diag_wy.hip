// The DIAG_WY form of the per-channel decay pre-pass (zoo_diag_prep.h)
#include "zoo_diag_prep.h"

int zoo_diag_wy_launch(const ZooDiagParams& p, int K, hipStream_t stream) { return zoo_diag::launch<DIAG_WY>(p, K, stream); }
