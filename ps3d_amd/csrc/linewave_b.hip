// linewave_b.hip -- wave line passes (linewave.hpp) of 90 to 150 points, n = A B: the
// physical values are the B elements of a lane, so B is the smaller factor (the x passes
// hold five or six fields of B elements).
#include "linewave.hpp"

namespace ps3d {

#define SIZES(X) X(90, 10, 9) X(96, 12, 8) X(100, 10, 10) X(108, 12, 9) X(120, 12, 10) X(144, 12, 12) X(150, 15, 10)
SIZES(PS3D_LW_TWO)
PS3D_LW_SET(b, SIZES)

}  // namespace ps3d
