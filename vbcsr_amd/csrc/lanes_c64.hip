// Lane-per-row SpMM kernels for c64 storage (see lanes.hpp).
#include "batched.hpp"
#include "lanes.hpp"
#include "quad_spmv.hpp"
#include "quads.hpp"
#include "smalls.hpp"
#include "tiles.hpp"

namespace vbh {
VBH_LANES_INSTANTIATE(c64, c64)
VBH_BATCHED_INSTANTIATE(c64, c64)
VBH_QUADS_INSTANTIATE(c64, c64)
VBH_SMALLS_INSTANTIATE(c64, c64)
VBH_SMALLS_ADJOINT_INSTANTIATE(c64)
VBH_TILES_INSTANTIATE(c64, c64)
VBH_TILES_ADJOINT_INSTANTIATE(c64)
VBH_QUAD_SPMV_INSTANTIATE(c64)
}  // namespace vbh
