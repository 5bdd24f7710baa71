// MFMA product for tensors of any size and alignment, fp16 operands.
#include "ptl_ragged.inc"

namespace ptl {
template int ragged<half_t>(RagArgs &, int, int, int, int);
template int ragged_deep<half_t>(const half_t *, const half_t *, half_t *, int, int, int, const half_t *);
}  // namespace ptl
