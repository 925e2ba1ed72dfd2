// The DIAG_GLA form of the per-channel decay pre-pass (zoo_diag_prep.h)
#include "zoo_diag_prep.h"

int zoo_diag_gla_launch(const ZooDiagParams& p, int K, hipStream_t stream) { return zoo_diag::launch<DIAG_GLA>(p, K, stream); }
