// Pass kernels for columns of 2^3 points (forward/inverse, intermediate/last).
#include "ntt_pass.hpp"

namespace pl {
PL_DEFINE_PASS_LAUNCHER(0)
}  // namespace pl
