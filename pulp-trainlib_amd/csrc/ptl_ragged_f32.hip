// MFMA product for tensors of any size and alignment, fp32 operands.
#include "ptl_ragged.inc"

namespace ptl {
template int ragged<float>(RagArgs &, int, int, int, int);
template int ragged_deep<float>(const float *, const float *, float *, int, int, int, const float *);
}  // namespace ptl
