// MFMA product for tensors of any size and alignment, fp16 operands.
#include "ptl_ragged.inc"

namespace ptl {
template int ragged<half_t>(RagArgs &, int, int, int, int);
}  // namespace ptl
