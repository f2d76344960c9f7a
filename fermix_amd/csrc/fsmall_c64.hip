// The LDS-resident LU / inverse and Parlett-Reid of field_small.inc for cx<float>.
#include "field_small.inc"

namespace fx {
FSMALL_INSTANTIATE(cx<float>)
}  // namespace fx
