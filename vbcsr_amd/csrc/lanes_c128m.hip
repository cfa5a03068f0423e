// Lane-per-row SpMM kernels for c128 vectors against c64 matrix values (see lanes.hpp).
#include "batched.hpp"
#include "lanes.hpp"
#include "quads.hpp"
#include "smalls.hpp"
#include "tiles.hpp"

namespace vbh {
VBH_LANES_INSTANTIATE(c128, c64)
VBH_BATCHED_INSTANTIATE(c128, c64)
VBH_QUADS_INSTANTIATE(c128, c64)
VBH_SMALLS_INSTANTIATE(c128, c64)
VBH_TILES_INSTANTIATE(c128, c64)
}  // namespace vbh
