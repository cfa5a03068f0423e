// Lane-per-row SpMM kernels for double vectors against float matrix values (see lanes.hpp).
#include "batched.hpp"
#include "lanes.hpp"
#include "quads.hpp"
#include "smalls.hpp"
#include "tiles.hpp"

namespace vbh {
VBH_LANES_INSTANTIATE(double, float)
VBH_BATCHED_INSTANTIATE(double, float)
VBH_QUADS_INSTANTIATE(double, float)
VBH_SMALLS_INSTANTIATE(double, float)
VBH_TILES_INSTANTIATE(double, float)
}  // namespace vbh
