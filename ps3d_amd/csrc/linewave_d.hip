// linewave_d.hip -- wave line passes (linewave.hpp) of 240 to 300 points, n = A B: the
// physical values are the B elements of a lane, so B is the smaller factor (the x passes
// hold five or six fields of B elements).
#include "linewave.hpp"

namespace ps3d {

#define SIZES(X) X(240, 16, 15) X(250, 25, 10) X(270, 18, 15) X(288, 18, 16) X(300, 20, 15)
SIZES(PS3D_LW_TWO)
PS3D_LW_SET(d, SIZES)

}  // namespace ps3d
