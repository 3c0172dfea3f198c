// linewave_c.hip -- wave line passes (linewave.hpp) of 160 to 216 points, n = A B: the
// physical values are the B elements of a lane, so B is the smaller factor (the x passes
// hold five or six fields of B elements).
#include "linewave.hpp"

namespace ps3d {

#define SIZES(X) X(160, 16, 10) X(162, 18, 9) X(180, 15, 12) X(192, 16, 12) X(200, 20, 10) X(216, 18, 12)
SIZES(PS3D_LW_TWO)
PS3D_LW_SET(c, SIZES)

}  // namespace ps3d
