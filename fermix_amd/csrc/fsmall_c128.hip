// The LDS-resident LU / inverse and Parlett-Reid of field_small.inc for cx<double>.
#include "field_small.inc"

namespace fx {
FSMALL_INSTANTIATE(cx<double>)
}  // namespace fx
