// Both gradients of a convolution in one launch, fp32.
#include "ptl_ragged_back.inc"

namespace ptl {
template RagBackPlan ragged_back_plan<float>(const RagProd *, const RagProd *, int, RagBack);
template int ragged_back<float>(RagConvArgs &, RagConvArgs &, const RagGeo *, RagBack, int, const RagBackPlan &);
}  // namespace ptl
