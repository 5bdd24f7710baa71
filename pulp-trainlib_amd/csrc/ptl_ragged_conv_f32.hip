// Convolutions as products with patch matrices, fp32.
#include "ptl_ragged_conv.inc"

namespace ptl {
template int ragged_conv<float>(RagConvArgs &, int, int, const RagPlan &);
template RagPlan ragged_conv_plan<float>(const RagProd *, int, int, int);
template int ragged_relay<float>(RagConvArgs &, const RagTurn *, int);
}  // namespace ptl
