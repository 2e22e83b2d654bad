// Tiled cost-volume kernels instantiated for double storage: forward, 1, 2 and 4 lanes per
// pixel and the entry points.
#define CHOP_S double
#define CHOP_TILED_FORWARD
#define CHOP_LPP_PART 0
#include "tiled_launch.inc"
