// Lane-per-row SpMM kernels for c128 storage (see lanes.hpp).
#include "batched.hpp"
#include "lanes.hpp"
#include "quad_spmv.hpp"
#include "quads.hpp"
#include "smalls.hpp"
#include "tiles.hpp"

namespace vbh {
VBH_LANES_INSTANTIATE(c128, c128)
VBH_BATCHED_INSTANTIATE(c128, c128)
VBH_QUADS_INSTANTIATE(c128, c128)
VBH_SMALLS_INSTANTIATE(c128, c128)
VBH_SMALLS_ADJOINT_INSTANTIATE(c128)
VBH_TILES_INSTANTIATE(c128, c128)
VBH_TILES_ADJOINT_INSTANTIATE(c128)
VBH_QUAD_SPMV_INSTANTIATE(c128)
}  // namespace vbh
