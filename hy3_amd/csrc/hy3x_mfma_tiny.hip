// hy3x_mfma_tiny.hip -- the 8-token shape of the MFMA grouped GEMMs: the same
// source as the narrow shape, compiled with HY3X_MFMA_TINY into namespace
// hy3x::mfma_tiny.
#define HY3X_MFMA_TINY
#include "hy3x_mfma.hip"
