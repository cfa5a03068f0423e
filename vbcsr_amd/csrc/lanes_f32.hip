// Lane-per-row SpMM kernels for float storage (see lanes.hpp).
#include "batched.hpp"
#include "lanes.hpp"
#include "quad_spmv.hpp"
#include "quads.hpp"
#include "smalls.hpp"
#include "tiles.hpp"

namespace vbh {
VBH_LANES_INSTANTIATE(float, float)
VBH_BATCHED_INSTANTIATE(float, float)
VBH_QUADS_INSTANTIATE(float, float)
VBH_SMALLS_INSTANTIATE(float, float)
VBH_SMALLS_ADJOINT_INSTANTIATE(float)
VBH_TILES_INSTANTIATE(float, float)
VBH_TILES_ADJOINT_INSTANTIATE(float)
VBH_QUAD_SPMV_INSTANTIATE(float)
}  // namespace vbh
