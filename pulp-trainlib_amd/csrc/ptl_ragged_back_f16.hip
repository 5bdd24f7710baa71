// Both gradients of a convolution in one launch, fp16.
#include "ptl_ragged_back.inc"

namespace ptl {
template RagBackPlan ragged_back_plan<half_t>(const RagProd *, const RagProd *, int, RagBack);
template int ragged_back<half_t>(RagConvArgs &, RagConvArgs &, const RagGeo *, RagBack, int, const RagBackPlan &);
}  // namespace ptl
