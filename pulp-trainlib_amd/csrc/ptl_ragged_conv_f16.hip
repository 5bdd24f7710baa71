// Convolutions as products with patch matrices, fp16.
#include "ptl_ragged_conv.inc"

namespace ptl {
template int ragged_conv<half_t>(RagConvArgs &, int, int, const RagPlan &);
template RagPlan ragged_conv_plan<half_t>(const RagProd *, int, int, int);
template int ragged_relay<half_t>(RagConvArgs &, const RagTurn *, int);
}  // namespace ptl
