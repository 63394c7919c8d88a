// faces_flow_g5.hip -- the one-item kernel's launches for n = 13, 14, 15, 16
// (faces_flow_launch.hpp), compiled apart from the other element sizes.
#include "faces_flow_launch.hpp"

namespace faces {

FACES_FLOW_GROUP(launch_flow_g5, FACES_FLOW_CASE(13) FACES_FLOW_CASE(14) FACES_FLOW_CASE(15) FACES_FLOW_CASE(16))

}  // namespace faces
