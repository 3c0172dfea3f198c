// linewave_e.hip -- wave line passes (linewave.hpp) of 320 to 384 points, n = A B: the
// physical values are the B elements of a lane, so B is the smaller factor (the x passes
// hold five or six fields of B elements).
#include "linewave.hpp"

namespace ps3d {

#define SIZES(X) X(320, 20, 16) X(324, 18, 18) X(360, 20, 18) X(384, 24, 16)
SIZES(PS3D_LW_TWO)
PS3D_LW_SET(e, SIZES)

}  // namespace ps3d
