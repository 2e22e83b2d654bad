// Tiled cost-volume kernels instantiated for double storage: backward, 8 and 16 lanes per
// pixel.
#define CHOP_S double
#define CHOP_TILED_BACKWARD
#define CHOP_LPP_PART 1
#include "tiled_launch.inc"
