// Lane-per-row SpMM kernels for double storage (see lanes.hpp).
#include "batched.hpp"
#include "lanes.hpp"
#include "quad_spmv.hpp"
#include "quads.hpp"
#include "smalls.hpp"
#include "tiles.hpp"

namespace vbh {
VBH_LANES_INSTANTIATE(double, double)
VBH_BATCHED_INSTANTIATE(double, double)
VBH_QUADS_INSTANTIATE(double, double)
VBH_SMALLS_INSTANTIATE(double, double)
VBH_SMALLS_ADJOINT_INSTANTIATE(double)
VBH_TILES_INSTANTIATE(double, double)
VBH_TILES_ADJOINT_INSTANTIATE(double)
VBH_QUAD_SPMV_INSTANTIATE(double)
}  // namespace vbh
