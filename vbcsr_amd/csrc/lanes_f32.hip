// Lane-per-row SpMM kernels for float storage (see lanes.hpp).
#include "lanes.hpp"
#include "quads.hpp"

namespace vbh {
VBH_LANES_INSTANTIATE(float, float)
VBH_QUADS_INSTANTIATE(float, float)
}  // namespace vbh
