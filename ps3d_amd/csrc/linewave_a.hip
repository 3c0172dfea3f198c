// linewave_a.hip -- wave line passes (linewave.hpp) of 16 to 80 points, n = A B: the
// physical values are the B elements of a lane, so B is the smaller factor (the x passes
// hold five or six fields of B elements).
#include "linewave.hpp"

namespace ps3d {

#define SIZES(X) X(16, 4, 4) X(18, 6, 3) X(20, 5, 4) X(24, 6, 4) X(30, 6, 5) X(32, 8, 4) X(36, 6, 6) X(40, 8, 5) X(48, 8, 6) X(50, 10, 5) X(54, 9, 6) X(60, 10, 6) X(72, 9, 8) X(80, 10, 8)
SIZES(PS3D_LW_TWO)
PS3D_LW_SET(a, SIZES)

}  // namespace ps3d
